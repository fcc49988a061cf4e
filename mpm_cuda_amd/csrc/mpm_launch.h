// mpm_launch.h -- host-side launchers of the step kernels.
#pragma once

#include "mpm_internal.h"

namespace mpm {

int launch_zero_u32(hipStream_t st, uint32_t *p, int n);
int launch_p2g_atomic(hipStream_t st, const GridP &g, const MatP &m, const PartView &pv, float dt,
                      int sweeps, int tau_stored, float4 *grid, uint32_t *flags, uint32_t *counters,
                      int threads);
int launch_count_active(hipStream_t st, const uint32_t *act, uint32_t seq, int64_t nblocks, uint32_t *counters,
                        const float4 *gv);
int launch_list_marked(hipStream_t st, const uint32_t *flags, int nblocks, uint32_t *list, uint32_t *counters);
int launch_list_near(hipStream_t st, const GridP &g, const int32_t *blk_tile, int ngroups, int nblocks, uint32_t *flags,
                     uint32_t *list, uint32_t *counters);
int launch_bsort_list(hipStream_t st, const SortSlice *tab, int ns, int wgs);
int launch_grid_update(hipStream_t st, const GridP &g, float dt, const uint32_t *list, uint32_t *flags, uint32_t *act,
                       uint32_t seq, uint32_t *counters, float4 *gmp, float4 *gv, int64_t nblocks,
                       const float4 *staging, const int32_t *blk_tile, int ngroups, uint32_t staging_cap,
                       uint32_t *host_count, uint32_t *host_seq, uint32_t launch, int clear_maxima);
// A G2P that applies a re-sort: slot j of po receives particle perm[j] of
// the view, its id (pid -> pid_out) and, with copy_q, its quaternion.
struct G2PMove {
    const uint32_t *perm;
    PartView po;
    const uint32_t *pid;
    uint32_t *pid_out;
    int copy_q;
};
int launch_g2p(hipStream_t st, const GridP &g, const MatP &m, const PartView &pv, float dt,
               const float4 *gv, int write_tau, int sweeps, uint32_t *counters, int threads,
               const G2PMove *mv = nullptr);
int launch_compute_tau(hipStream_t st, const MatP &m, const PartView &pv, int sweeps, uint32_t *counters);
int launch_p2g_spill(hipStream_t st, const GridP &g, const MatP &m, const PartView &pv, float dt,
                     const uint32_t *list, uint32_t list_cap, uint32_t *counters, float4 *grid, uint32_t *flags, uint32_t *blocks,
                     uint32_t *host_count, uint32_t *host_seq, uint32_t seq);
int launch_dt_scan(hipStream_t st, const MatP &m, const PartView &pv, uint32_t *counters);
int launch_dt_clear(hipStream_t st, uint32_t *counters);
int launch_dt_control(hipStream_t st, const DtRule &rule, uint32_t *counters);

// FAST form (mpm_fast.hip)
int fast_prepare(mpm_sim *s);                 // (re)sort particles and build P2G tiles when due
int launch_p2g_tiles(mpm_sim *s, float dt);
int spill_publish(mpm_sim *s, uint32_t **count, uint32_t **seq, uint32_t *launch);   // where the grid phase writes its count
int launch_g2p_fast(mpm_sim *s, float dt);
int launch_g2p_groups(hipStream_t st, const G2PArgs &a, uint32_t wgs, int threads, bool move);
int launch_g2p2g(mpm_sim *s, int group, float dt, float dt_next);   // FUSED form
int sort_all(mpm_sim *s, bool defer = false);  // sort every group now and rebuild the tiles
int sort_for_g2p(mpm_sim *s);                 // a due re-sort, applied by the coming FAST G2P
int finish_g2p_move(mpm_sim *s, bool moved);  // after that G2P (or instead of it): the particles in the new order
int fast_ready(mpm_sim *s);                   // sorted once, stored stress current
PartView view_of(mpm_sim *s, int g);

// Batched stages over a BatchSlice table in device memory (mpm_step.hip,
// mpm_fast.hip); host side in mpm_batch.hip.
void fill_batch_slice(mpm_sim *s, BatchSlice &b);
// Batched re-sort (mpm_fast.hip): launch sizes of a set of scenes, one
// scene's table entry in its current parity, and the launches.
struct SortBatchPlan {
    int passes = 0, tiles = 0, spine = 0, runs = 0, scan = 0, emit = 0, rank = 0;
};
void sort_batch_plan(mpm_sim *const *sims, int ns, SortBatchPlan &pl);
int fill_sort_slice(mpm_sim *s, SortSlice &t);
int launch_sort_batch(hipStream_t st, const SortSlice *tab, int ns, const SortBatchPlan &pl);
// Warm-start particle lists of a simulator (mpm_api.hip).
int ensure_warm_lists(mpm_sim *s);
int launch_p2g_batch(hipStream_t st, int mats, const BatchSlice *tab, int nslices, int wgs);
// Planes of w floats (plane c at planes + c * stride) of n particles to the
// host rows out[id][w]; ids NULL: in stored order, else `scratch` holds n * w
// floats rounded up to 16 bytes (mpm_read.hip).
int read_rows(ReadStage &rs, hipStream_t st, const float *planes, int64_t stride, int64_t n, int w,
              const uint32_t *ids, float *scratch, float *out);
bool tile_shape_valid(int tile);              // values of mpm_config.tile and mpm_batch_shape.p2g_tile
int launch_permute_batch(hipStream_t st, const BatchSlice *src, const BatchSlice *dst, int nslices, int wgs);
int launch_grid_batch(hipStream_t st, const BatchSlice *tab, int nslices, int wgs);
int launch_g2p_batch(hipStream_t st, int mats, const BatchSlice *tab, int nslices, int wgs, int threads);
int launch_mlp_infer(hipStream_t st, const float *params, const PartView &pv);
int launch_mlp_infer_batch(hipStream_t st, const float *params, const BatchSlice *tab, int nslices, int group,
                           int64_t chunks);

// Scene sampling and files (scene.cpp)
int sample_object(const mpm_config &cfg, const mpm_object &obj, std::vector<float> &xyz);
int write_bgeo(const char *path, const float *xyz, int64_t n);

}  // namespace mpm
