// mpm_batch.hip -- many independent scenes advanced together.
//
// No counterpart in the reference (it steps one MPMSimulator per process).
// Each scene is an mpm_sim with one particle group in the FAST form.  The
// batch keeps a table of the scenes' parameters (BatchSlice) in device memory
// and advances every scene by one step with one launch per stage -- P2G tiles
// (per 64 scenes), grid update, G2P -- each over the scenes of all materials,
// plus one warm-start inference launch per set of scenes with equal network
// weights.  (16 scenes of the three materials, 0.9M particles, 48 steps: 6.3 ms
// with a hipGraph of one branch per material joined at every step, 5.9 with a
// graph of these three launches, 5.7 launched directly.)  A longer run of more
// particles takes two such chains of launches, each over half of the scenes
// (make_chains).
// Every `sort_every` steps all scenes are re-sorted, one launch per stage of
// the sort, replayed as a hipGraph.  Sorting moves particle storage between
// two buffers, so there is one graph per buffer parity.  Launch widths come
// from mpm_batch_autotune, which times the candidates of each stage on live
// steps; results do not depend on them (every tile, block and particle is
// processed by exactly one workgroup).
#include "mpm_launch.h"

#include <string.h>

#include <algorithm>
#include <vector>

using namespace mpm;

namespace {

constexpr int NCAND = 4;
const int P2G_CAND[NCAND] = {1024, 2048, 4096, 8192};   // workgroups of four waves
const int GRID_CAND[NCAND] = {1024, 2048, 4096, 8192};
const int G2P_CAND[NCAND] = {64, 128, 192, 256};
constexpr int NTILE = 3;
const int TILE_CAND[NTILE] = {256, 384, 512};            // values of p2g_tile; the P2G is the same with each

// What the tables and the captured graphs depend on, per scene.
struct SceneSig {
    float *P0, *P1;
    uint32_t *pid0, *pid1;
    float *mlp_w;
    int64_t mlp_version;
    int warm;
    double dt;
    int sweeps;
    bool operator==(const SceneSig &o) const
    {
        return P0 == o.P0 && P1 == o.P1 && pid0 == o.pid0 && pid1 == o.pid1 && mlp_w == o.mlp_w &&
               mlp_version == o.mlp_version && warm == o.warm && dt == o.dt && sweeps == o.sweeps;
    }
};

// Scenes [begin, begin + count) of the tables, whose steps follow one another
// on one stream.
struct Chain {
    int begin, count;
    int mats;                           // their material, MAT_ANY: several
    hipStream_t stream;                 // null: the batch's own
    hipEvent_t done;
    std::vector<std::pair<int, int64_t>> warm;      // weight sets among them, 64-particle chunks of each
    SortBatchPlan sort;                 // their re-sort, and the workgroups of its move
    int permute_wgs;
    hipGraphExec_t sort_exec[2];        // per parity
};

}  // namespace

struct mpm_batch {
    std::vector<mpm_sim *> sims;
    hipStream_t stream = nullptr;
    mpm_batch_shape shape{};
    // particle buffers of parity 0 / 1 (P, P_alt of each scene at creation)
    std::vector<float *> P0, P1;
    std::vector<uint32_t *> pid0, pid1;
    BatchSlice *tab[2] = {};
    std::vector<SceneSig> sig;          // signature the tables and graphs were built for
    bool built = false;
    int parity = 0;
    int64_t steps_since_sort = 0;
    int64_t total = 0;
    Chain all{};                        // every scene, on the batch's stream
    std::vector<Chain> chains;          // two halves side by side (see make_chains), or all
    bool forked = false;                // the chains' streams are ahead of the batch's
    SortSlice *stab[2] = {};            // batched re-sort tables of both parities
    // warm-start weight sets: scenes with equal weights share one inference launch
    std::vector<const float *> warm_params; // device weights of each set
    std::vector<int> warm_group;            // per scene, -1: cold
    hipEvent_t ev_done = nullptr, ev_fork = nullptr;
    std::vector<hipEvent_t> ev_join;
    std::vector<hipEvent_t> tev;        // step timing events
};

namespace {

bool warm_on(const mpm_sim *s)
{
    return s->cfg.warm_start == MPM_WARM_MLP && s->mlp_w && s->mlp_count == mpm_mlp_param_count() &&
           s->groups[0].mat.type != MPM_WATER;
}

SceneSig sig_of(const mpm_batch *b, size_t k)
{
    const mpm_sim *s = b->sims[k];
    return SceneSig{b->P0[k], b->P1[k], b->pid0[k], b->pid1[k], s->mlp_w, s->mlp_version, warm_on(s) ? 1 : 0,
                    s->cfg.dt, s->cfg.svd_sweeps};
}

int parity_of(const mpm_batch *b, size_t k)
{
    const mpm_sim *s = b->sims[k];
    if (s->P == b->P0[k] && s->P_alt == b->P1[k]) return 0;
    if (s->P == b->P1[k] && s->P_alt == b->P0[k]) return 1;
    return -1;
}

// Point the scene's host view at the buffers of parity p.
void set_parity(mpm_batch *b, size_t k, int p)
{
    mpm_sim *s = b->sims[k];
    s->P = p ? b->P1[k] : b->P0[k];
    s->P_alt = p ? b->P0[k] : b->P1[k];
    s->pid = p ? b->pid1[k] : b->pid0[k];
    s->pid_alt = p ? b->pid0[k] : b->pid1[k];
}

// G2P workgroups of a chain's scenes.
int g2p_wgs(const mpm_batch *b, const Chain &c, int threads)
{
    uint32_t w = 0;
    for (int k = c.begin; k < c.begin + c.count; ++k)
        w += (uint32_t)((b->sims[k]->groups[0].n + threads - 1) / threads);
    return (int)round_xcd(w);
}

int check(int rc, const char *what) { return rc ? hip_fail((hipError_t)rc, what) : MPM_OK; }

// One step of a chain's scenes (parity p tables): P2G, grid update, the
// warm-start inference of each weight set, G2P.  With `ev` (STEP_EVENTS, the
// autotuner's stage timing) an event before the first stage and after each.
constexpr int STEP_EVENTS = 5, STAGE_BEGIN[3] = {0, 1, 3};      // P2G, grid update, G2P end at the next one
int enqueue_step(mpm_batch *b, const Chain &c, int p, int p2g, int grid, int g2p_threads, hipEvent_t *ev)
{
    hipStream_t st = c.stream ? c.stream : b->stream;
    const BatchSlice *tab = b->tab[p] + c.begin;
    int rc;
    if (ev) MPM_HIP(hipEventRecord(ev[0], st));
    if ((rc = check(launch_p2g_batch(st, c.mats, tab, c.count, p2g), "p2g_batch"))) return rc;
    if (ev) MPM_HIP(hipEventRecord(ev[1], st));
    if ((rc = check(launch_grid_batch(st, tab, c.count, grid), "grid_batch"))) return rc;
    if (ev) MPM_HIP(hipEventRecord(ev[2], st));
    for (const auto &w : c.warm)
        if ((rc = check(launch_mlp_infer_batch(st, b->warm_params[w.first], tab, c.count, w.first, w.second),
                        "mlp_infer_batch")))
            return rc;
    if (ev) MPM_HIP(hipEventRecord(ev[3], st));
    const int wgs = g2p_wgs(b, c, g2p_threads);
    if (wgs && (rc = check(launch_g2p_batch(st, c.mats, tab, c.count, wgs, g2p_threads), "g2p_batch"))) return rc;
    if (ev) MPM_HIP(hipEventRecord(ev[4], st));
    return MPM_OK;
}

// The chains' streams go on after the batch's, and the batch's after theirs.
int fork_chains(mpm_batch *b)
{
    if (b->forked || b->chains.size() < 2) return MPM_OK;
    MPM_HIP(hipEventRecord(b->ev_fork, b->stream));
    for (Chain &c : b->chains)
        if (c.stream) MPM_HIP(hipStreamWaitEvent(c.stream, b->ev_fork, 0));
    b->forked = true;
    return MPM_OK;
}

int join_chains(mpm_batch *b)
{
    if (!b->forked) return MPM_OK;
    b->forked = false;
    for (Chain &c : b->chains)
        if (c.stream) {
            MPM_HIP(hipEventRecord(c.done, c.stream));
            MPM_HIP(hipStreamWaitEvent(b->stream, c.done, 0));
        }
    return MPM_OK;
}

// Re-sort a chain's scenes from parity p into parity 1 - p: keys, order and
// tiles of all of them with one launch per sort stage, then one launch moves
// every scene's particles into the parity 1 - p buffers in its new order (the
// warm-start lists, which name old slots, are dropped).  The caller points the
// host views at parity 1 - p.
int enqueue_sort(mpm_batch *b, const Chain &c, hipStream_t st, int p)
{
    int rc = launch_sort_batch(st, b->stab[p] + c.begin, c.count, c.sort);
    if (rc) return rc;
    return check(launch_permute_batch(st, b->tab[p] + c.begin, b->tab[p ^ 1] + c.begin, c.count, c.permute_wgs),
                 "permute_batch");
}

void drop_graphs(mpm_batch *b)
{
    auto drop = [](Chain &c) {
        for (int p = 0; p < 2; ++p) {
            if (c.sort_exec[p]) (void)hipGraphExecDestroy(c.sort_exec[p]);
            c.sort_exec[p] = nullptr;
        }
    };
    drop(b->all);
    for (Chain &c : b->chains) drop(c);
}

// The graph of a chain's re-sort from parity p, at its first use.
int capture_sort(mpm_batch *b, Chain &c, int p)
{
    MPM_HIP(hipStreamBeginCapture(b->stream, hipStreamCaptureModeRelaxed));
    int rc = enqueue_sort(b, c, b->stream, p);
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture(b->stream, &graph);
    if (rc) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc;
    }
    if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
    e = hipGraphInstantiate(&c.sort_exec[p], graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) return hip_fail(e, "hipGraphInstantiate");
    return MPM_OK;
}

// Warm scenes grouped by identical weights.
void group_warm(mpm_batch *b)
{
    b->warm_params.clear();
    b->warm_group.assign(b->sims.size(), -1);
    std::vector<size_t> rep;                        // first scene of each set
    for (size_t k = 0; k < b->sims.size(); ++k) {
        mpm_sim *s = b->sims[k];
        if (!warm_on(s)) continue;
        int g = -1;
        for (size_t r = 0; r < rep.size() && g < 0; ++r)
            if (b->sims[rep[r]]->mlp_host == s->mlp_host) g = (int)r;
        if (g < 0) {
            g = (int)rep.size();
            rep.push_back(k);
            b->warm_params.push_back(s->mlp_w);
        }
        b->warm_group[k] = g;
    }
    auto sets = [&](Chain &c) {
        std::vector<int64_t> chunks(rep.size(), 0);
        for (int k = c.begin; k < c.begin + c.count; ++k)
            if (b->warm_group[k] >= 0) chunks[b->warm_group[k]] += (b->sims[k]->groups[0].n + 63) / 64;
        c.warm.clear();
        for (size_t g = 0; g < chunks.size(); ++g)
            if (chunks[g]) c.warm.push_back({(int)g, chunks[g]});
    };
    sets(b->all);
    for (Chain &c : b->chains) sets(c);
}

// Device tables for both parities.
int build(mpm_batch *b)
{
    const size_t n = b->sims.size();
    MPM_HIP(hipStreamSynchronize(b->stream));       // no replay still reads the tables
    group_warm(b);
    for (mpm_sim *s : b->sims) {
        int rc = warm_on(s) ? ensure_warm_lists(s) : MPM_OK;
        if (rc) return rc;
        // the re-sort order the batched move reads (allocated here, never
        // inside a captured sort)
        if (s->g2p_perm_cap < s->cap) {
            if (s->g2p_perm) (void)hipFree(s->g2p_perm);
            s->g2p_perm = nullptr;
            s->g2p_perm_cap = 0;
            MPM_HIP(hipMalloc(&s->g2p_perm, (size_t)s->cap * sizeof(uint32_t)));
            s->g2p_perm_cap = s->cap;
        }
    }
    for (int p = 0; p < 2; ++p) {
        std::vector<BatchSlice> h(n);
        for (size_t k = 0; k < n; ++k) {
            mpm_sim *s = b->sims[k];
            float *P = s->P, *Pa = s->P_alt;
            uint32_t *id = s->pid, *ida = s->pid_alt;
            set_parity(b, k, p);
            fill_batch_slice(s, h[k]);
            h[k].mat.warm_sweeps = warm_on(s) ? std::max(1, s->cfg.warm_sweeps) : 0;
            h[k].warm_group = b->warm_group[k];
            if (warm_on(s)) {
                // the G2P lists the particles that take the SVD; the next
                // step's inference runs over them (k_grid_batch hands them over)
                h[k].mat.wlist = s->warm_list;
                h[k].mat.wcount = s->warm_cnt + 1;
                h[k].warm_cnt = s->warm_cnt;
            }
            s->P = P; s->P_alt = Pa; s->pid = id; s->pid_alt = ida;
        }
        MPM_HIP(hipMemcpy(b->tab[p], h.data(), n * sizeof(BatchSlice), hipMemcpyHostToDevice));
        std::vector<SortSlice> hs(n);
        for (size_t k = 0; k < n; ++k) {
            mpm_sim *s = b->sims[k];
            float *P = s->P, *Pa = s->P_alt;
            uint32_t *id = s->pid, *ida = s->pid_alt;
            set_parity(b, k, p);
            int rc = fill_sort_slice(s, hs[k]);
            s->P = P; s->P_alt = Pa; s->pid = id; s->pid_alt = ida;
            if (rc) return rc;
        }
        MPM_HIP(hipMemcpy(b->stab[p], hs.data(), n * sizeof(SortSlice), hipMemcpyHostToDevice));
    }
    b->sig.clear();
    for (size_t k = 0; k < n; ++k) b->sig.push_back(sig_of(b, k));
    drop_graphs(b);
    b->built = true;
    return MPM_OK;
}

// Waits for *flag, `ticks` of the 100 MHz clock at most.
__global__ void k_wait_flag(const uint32_t *flag, uint32_t *seen, long long ticks)
{
    const long long t0 = wall_clock64();
    while (!__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        if (wall_clock64() - t0 > ticks) return;
        __builtin_amdgcn_s_sleep(8);
    }
    *seen = 1u;
}
__global__ void k_set_flag(uint32_t *flag) { __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Whether kernels of the two streams run at the same time: not where the
// streams share a hardware queue, whose kernels then take turns at ~25 us each.
int streams_overlap(hipStream_t a, hipStream_t b, uint32_t *words, bool &yes)
{
    uint32_t seen = 0;
    if (int rc = check(launch_zero_u32(a, words, 2), "zero")) return rc;
    MPM_HIP(hipStreamSynchronize(a));
    hipLaunchKernelGGL(k_wait_flag, dim3(1), dim3(1), 0, a, words, words + 1, 50000ll);      // 0.5 ms
    hipLaunchKernelGGL(k_set_flag, dim3(1), dim3(1), 0, b, words);
    MPM_HIP(hipGetLastError());
    MPM_HIP(hipStreamSynchronize(b));
    MPM_HIP(hipStreamSynchronize(a));
    MPM_HIP(hipMemcpy(&seen, words + 1, 4, hipMemcpyDeviceToHost));
    yes = seen != 0u;
    return MPM_OK;
}

Chain chain_of(const mpm_batch *b, int begin, int end)
{
    Chain c{begin, end - begin, -1, nullptr, nullptr, {}, {}, 0, {nullptr, nullptr}};
    uint32_t wgs = 0;
    for (int k = begin; k < end; ++k) {
        const int t = b->sims[k]->groups[0].mat.type;
        c.mats = c.mats < 0 || c.mats == t ? t : MAT_ANY;
        wgs += (uint32_t)((b->sims[k]->groups[0].n + 255) / 256);
    }
    c.permute_wgs = (int)round_xcd(wgs);
    sort_batch_plan(b->sims.data() + begin, end - begin, c.sort);
    return c;
}

// Two chains of about equal particles on streams that overlap, joined only at
// the end of a run: one's launch tails, gather latencies and re-sort beside the
// other's LDS work.  ms a step with one chain and two: 64 scenes, 8.7M
// particles 1.013 and 0.898 (0.925 with the materials as branches of a graph,
// joined at each step; 0.912 with a join at each re-sort); 16 scenes, 1.9M 0.233
// and 0.204; 3 scenes, 0.43M 0.075 and 0.069; 4 scenes, 0.2M 0.051 and 0.047.
// Three chains: 0.89, 0.204 and no better than one below 1M.  Fewer particles
// are the host's launches either way.  A fork and a join cost ~20 us, so a run
// of a few steps takes one chain.
constexpr int64_t CHAIN_PARTICLES = 200000;
constexpr int32_t CHAIN_STEPS = 12;
int make_chains(mpm_batch *b)
{
    const int n = (int)b->sims.size();
    b->all = chain_of(b, 0, n);
    b->chains = {b->all};
    if (n < 2 || b->total < CHAIN_PARTICLES) return MPM_OK;
    int cut = 0;
    for (int64_t sum = 0; cut < n - 1 && sum < b->total / 2; ++cut) sum += b->sims[cut]->groups[0].n;
    uint32_t *words = nullptr;
    MPM_HIP(hipMalloc(&words, 8));
    std::vector<hipStream_t> tried;     // kept until the end: a queue is given to the next stream in turn
    int rc = MPM_OK;
    bool yes = false;
    while (!rc && !yes && tried.size() < 4) {
        hipStream_t st = nullptr;
        const hipError_t e = hipStreamCreateWithFlags(&st, hipStreamNonBlocking);
        if (e != hipSuccess) { rc = hip_fail(e, "stream"); break; }
        tried.push_back(st);
        rc = streams_overlap(b->stream, st, words, yes);
    }
    (void)hipFree(words);
    if (!rc && yes) {
        b->chains = {chain_of(b, 0, cut), chain_of(b, cut, n)};
        b->chains[1].stream = tried.back();
        tried.pop_back();
        hipError_t e = hipEventCreateWithFlags(&b->chains[1].done, hipEventDisableTiming);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&b->ev_fork, hipEventDisableTiming);
        if (e != hipSuccess) rc = hip_fail(e, "event");
    }
    for (hipStream_t st : tried) (void)hipStreamDestroy(st);
    return rc;
}

int validate_shape(const mpm_batch_shape &s)
{
    if (s.p2g_workgroups < 1 || s.p2g_workgroups > (1 << 20)) return set_error(MPM_ERR_INVALID, "p2g_workgroups out of range");
    if (s.grid_workgroups < 1 || s.grid_workgroups > (1 << 20)) return set_error(MPM_ERR_INVALID, "grid_workgroups out of range");
    if (s.g2p_threads < 64 || s.g2p_threads > 256 || s.g2p_threads % 64)
        return set_error(MPM_ERR_INVALID, "g2p_threads must be 64, 128, 192 or 256");
    if (s.sort_every < 1) return set_error(MPM_ERR_INVALID, "sort_every must be >= 1");
    if (s.p2g_tile != 0 && !tile_shape_valid(s.p2g_tile)) return set_error(MPM_ERR_INVALID, "p2g_tile must be 256, 384 or 512");
    return MPM_OK;
}

// Before a run: every scene in one buffer parity with a valid stress, the
// tables and graphs current, and the batch stream after the scenes' streams.
int prepare(mpm_batch *b)
{
    const size_t n = b->sims.size();
    if (int rc = join_chains(b)) return rc;         // of a run that ended early
    for (size_t k = 0; k < n; ++k) {
        mpm_sim *s = b->sims[k];
        if (!s->counters_clean)         // a batch's grid update leaves it cleared
            if (int rc = check(launch_zero_u32(s->stream, s->counters + CT_SPILL, 1), "zero")) return rc;
        s->counters_clean = true;
        s->spill_unread = false;
        if (parity_of(b, k) < 0) return set_error(MPM_ERR_INVALID, "a scene's particle storage changed since mpm_batch_create");
        if (s->groups.size() != 1) return set_error(MPM_ERR_INVALID, "a scene of the batch gained a particle group");
        int rc = fast_ready(s);
        if (rc) return rc;
    }
    // scenes stepped on their own may have re-sorted an odd number of times
    int ones = 0;
    for (size_t k = 0; k < n; ++k) ones += parity_of(b, k);
    b->parity = 2 * ones > (int)n ? 1 : 0;
    for (size_t k = 0; k < n; ++k)
        if (parity_of(b, k) != b->parity) {
            int rc = sort_all(b->sims[k]);
            if (rc) return rc;
        }
    bool same = b->built && b->sig.size() == n;
    for (size_t k = 0; same && k < n; ++k) same = sig_of(b, k) == b->sig[k];
    if (!same) {
        for (mpm_sim *s : b->sims) MPM_HIP(hipStreamSynchronize(s->stream));
        int rc = build(b);
        if (rc) return rc;
    }
    b->steps_since_sort = 0;
    for (mpm_sim *s : b->sims) b->steps_since_sort = std::max(b->steps_since_sort, s->steps_since_sort);
    for (size_t k = 0; k < n; ++k) {
        MPM_HIP(hipEventRecord(b->ev_join[k], b->sims[k]->stream));
        MPM_HIP(hipStreamWaitEvent(b->stream, b->ev_join[k], 0));
    }
    return MPM_OK;
}

// Scene streams continue after the batch's work.
int release(mpm_batch *b)
{
    MPM_HIP(hipEventRecord(b->ev_done, b->stream));
    for (mpm_sim *s : b->sims) MPM_HIP(hipStreamWaitEvent(s->stream, b->ev_done, 0));
    return MPM_OK;
}

void after_sort(mpm_batch *b)
{
    b->parity ^= 1;
    for (size_t k = 0; k < b->sims.size(); ++k) {
        mpm_sim *s = b->sims[k];
        set_parity(b, k, b->parity);
        s->sorted_valid = true;
        s->steps_since_sort = 0;
        s->sorted_at_launch = s->tile_launches;
        s->sorts += 1;
    }
    b->steps_since_sort = 0;
}

void after_step(mpm_batch *b)
{
    for (mpm_sim *s : b->sims) {
        s->steps += 1;
        s->time += s->cfg.dt;
        s->last_dt = s->cfg.dt;
        s->steps_since_sort += 1;
        s->tau_valid = true;
        s->last_phase = MPM_PHASE_G2P;
        s->act_seq = BATCH_SEQ;
    }
    b->steps_since_sort += 1;
}

// Sort when due (by graphs with `graphs`), then one step: with `chains` each
// chain on its stream, else all scenes together on the batch's.
int one_step(mpm_batch *b, int p2g, int grid, int g2p_threads, hipEvent_t *ev, bool graphs, bool chains)
{
    if (chains)
        if (int rc = fork_chains(b)) return rc;
    if (b->steps_since_sort >= b->shape.sort_every) {
        Chain *first = chains ? b->chains.data() : &b->all;
        for (Chain *c = first; c < first + (chains ? b->chains.size() : 1); ++c) {
            hipStream_t st = c->stream ? c->stream : b->stream;
            if (!graphs) {
                if (int rc = enqueue_sort(b, *c, st, b->parity)) return rc;
                continue;
            }
            if (!c->sort_exec[b->parity])
                if (int rc = capture_sort(b, *c, b->parity)) return rc;
            MPM_HIP(hipGraphLaunch(c->sort_exec[b->parity], st));
        }
        after_sort(b);
    }
    int rc = MPM_OK;
    if (!chains) {
        rc = enqueue_step(b, b->all, b->parity, p2g, grid, g2p_threads, ev);
    } else {
        for (size_t k = 0; k < b->chains.size() && !rc; ++k)
            rc = enqueue_step(b, b->chains[k], b->parity, p2g, grid, g2p_threads, nullptr);
    }
    if (rc) return rc;
    after_step(b);
    return MPM_OK;
}

hipEvent_t *timing_events(mpm_batch *b, size_t need)
{
    while (b->tev.size() < need) {
        hipEvent_t e = nullptr;
        if (hipEventCreate(&e) != hipSuccess) return nullptr;
        b->tev.push_back(e);
    }
    return b->tev.data();
}

}  // namespace

extern "C" {

void mpm_batch_shape_default(mpm_batch_shape *s)
{
    if (!s) return;
    memset(s, 0, sizeof *s);
    s->p2g_workgroups = 4096;
    s->grid_workgroups = 4096;
    s->g2p_threads = 256;
    s->sort_every = 24;
    s->use_graph = 1;
    s->p2g_tile = 384;
}

int mpm_batch_create(mpm_sim *const *sims, int32_t n, const mpm_batch_shape *shape, mpm_batch **out)
{
    if (!sims || !out) return set_error(MPM_ERR_INVALID, "null argument");
    *out = nullptr;
    if (n < 1 || n > BATCH_MAX) return set_error(MPM_ERR_INVALID, "a batch holds 1 to 256 scenes");
    mpm_batch_shape sh;
    mpm_batch_shape_default(&sh);
    if (shape) sh = *shape;
    int rc = validate_shape(sh);
    if (rc) return rc;
    for (int k = 0; k < n; ++k) {
        mpm_sim *s = sims[k];
        if (!s) return set_error(MPM_ERR_INVALID, "scene is null");
        if (s->cfg.form != MPM_FORM_FAST) return set_error(MPM_ERR_INVALID, "batched scenes use the FAST form");
        if (s->cfg.dt_mode != MPM_DT_FIXED)
            return set_error(MPM_ERR_INVALID, "batched scenes step with their fixed dt (dt_mode FIXED)");
        if (s->groups.size() != 1 || s->groups[0].n <= 0)
            return set_error(MPM_ERR_INVALID, "a batched scene holds exactly one non-empty particle group");
        for (int j = 0; j < k; ++j)
            if (sims[j] == s) return set_error(MPM_ERR_INVALID, "a scene appears twice in the batch");
    }
    mpm_batch *b = new mpm_batch();
    b->sims.assign(sims, sims + n);
    // ordered by material (stable): a chain then holds as few as may be
    std::stable_sort(b->sims.begin(), b->sims.end(), [](const mpm_sim *x, const mpm_sim *y) {
        return x->groups[0].mat.type < y->groups[0].mat.type;
    });
    b->shape = sh;
    auto fail = [&](int code) { mpm_batch_destroy(b); return code; };
    for (mpm_sim *s : b->sims) {
        if ((rc = fast_ready(s))) return fail(rc);         // buffers, first sort, stress
        b->total += s->groups[0].n;
    }
    for (mpm_sim *s : b->sims)
        if (hipStreamSynchronize(s->stream) != hipSuccess) return fail(hip_fail(hipErrorUnknown, "scene sync"));
    for (mpm_sim *s : b->sims) {
        b->P0.push_back(s->P); b->P1.push_back(s->P_alt);
        b->pid0.push_back(s->pid); b->pid1.push_back(s->pid_alt);
    }
    hipError_t e;
    if ((e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking)) != hipSuccess) return fail(hip_fail(e, "stream"));
    if ((e = hipMalloc(&b->tab[0], n * sizeof(BatchSlice))) != hipSuccess) return fail(hip_fail(e, "hipMalloc"));
    if ((e = hipMalloc(&b->tab[1], n * sizeof(BatchSlice))) != hipSuccess) return fail(hip_fail(e, "hipMalloc"));
    for (int p = 0; p < 2; ++p)
        if ((e = hipMalloc(&b->stab[p], n * sizeof(SortSlice))) != hipSuccess) return fail(hip_fail(e, "hipMalloc"));
    if ((e = hipEventCreateWithFlags(&b->ev_done, hipEventDisableTiming)) != hipSuccess) return fail(hip_fail(e, "event"));
    b->ev_join.assign(n, nullptr);
    for (auto &ev : b->ev_join)
        if ((e = hipEventCreateWithFlags(&ev, hipEventDisableTiming)) != hipSuccess) return fail(hip_fail(e, "event"));
    if ((rc = make_chains(b))) return fail(rc);
    *out = b;
    return MPM_OK;
}

int mpm_batch_get_shape(const mpm_batch *b, mpm_batch_shape *out)
{
    if (!b || !out) return set_error(MPM_ERR_INVALID, "null argument");
    *out = b->shape;
    return MPM_OK;
}

int mpm_batch_set_shape(mpm_batch *b, const mpm_batch_shape *shape)
{
    if (!b || !shape) return set_error(MPM_ERR_INVALID, "null argument");
    int rc = validate_shape(*shape);
    if (rc) return rc;
    b->shape = *shape;
    return MPM_OK;
}

int64_t mpm_batch_particles(const mpm_batch *b) { return b ? b->total : 0; }
int32_t mpm_batch_scenes(const mpm_batch *b) { return b ? (int32_t)b->sims.size() : 0; }

int mpm_batch_run(mpm_batch *b, int32_t nsteps, float *step_ms)
{
    if (!b) return set_error(MPM_ERR_INVALID, "batch is null");
    if (nsteps < 0) return set_error(MPM_ERR_INVALID, "nsteps must be >= 0");
    if (nsteps == 0) return MPM_OK;
    int rc = prepare(b);
    if (rc) return rc;
    // a step ends where the last of its chains' does: an event per chain after
    // each (the batch's stream first), all timed from the start
    const bool chains = b->chains.size() > 1 && nsteps >= CHAIN_STEPS;
    const size_t per = step_ms ? (chains ? b->chains.size() : 1) : 0;
    hipEvent_t *ev = per ? timing_events(b, (size_t)nsteps * per + 1) : nullptr;
    if (per && !ev) return set_error(MPM_ERR_HIP, "hipEventCreate failed");
    const bool graphs = b->shape.use_graph != 0;
    if (ev) MPM_HIP(hipEventRecord(ev[0], b->stream));
    for (int32_t k = 0; k < nsteps; ++k) {
        rc = one_step(b, b->shape.p2g_workgroups, b->shape.grid_workgroups, b->shape.g2p_threads, nullptr, graphs, chains);
        if (rc) return rc;
        for (size_t c = 0; c < per; ++c)
            MPM_HIP(hipEventRecord(ev[1 + k * per + c], c ? b->chains[c].stream : b->stream));
    }
    if ((rc = join_chains(b))) return rc;
    if ((rc = release(b))) return rc;
    if (ev) {
        MPM_HIP(hipStreamSynchronize(b->stream));
        float before = 0.0f;
        for (int32_t k = 0; k < nsteps; ++k) {
            float end = before;
            for (size_t c = 0; c < per; ++c) {
                float t = 0.0f;
                MPM_HIP(hipEventElapsedTime(&t, ev[0], ev[1 + k * per + c]));
                end = std::max(end, t);
            }
            step_ms[k] = end - before;
            before = end;
        }
    }
    return MPM_OK;
}

// Times each stage's launch-width candidates on live steps (rounds of
// NCAND steps, candidate c in step c of every round) and keeps the fastest
// median per stage; then, with those widths, the values of p2g_tile (rounds of
// NTILE steps; they select the same kernel) and keeps the fastest.  Advances every scene by
// reps * (NCAND + NTILE) steps.  ms_out (optional, 3 x NCAND + NTILE):
// median milliseconds of P2G, grid update and G2P per width candidate, then
// of P2G per p2g_tile.
int mpm_batch_autotune(mpm_batch *b, int32_t reps, float *ms_out)
{
    if (!b) return set_error(MPM_ERR_INVALID, "batch is null");
    if (reps < 1 || reps > 1000) return set_error(MPM_ERR_INVALID, "reps out of range [1,1000]");
    int rc = prepare(b);
    if (rc) return rc;
    const size_t per = STEP_EVENTS;
    hipEvent_t *ev = timing_events(b, (size_t)reps * (NCAND + NTILE) * per);
    if (!ev) return set_error(MPM_ERR_HIP, "hipEventCreate failed");
    for (int32_t r = 0; r < reps; ++r)
        for (int c = 0; c < NCAND; ++c) {
            hipEvent_t *e = ev + ((size_t)r * NCAND + c) * per;
            rc = one_step(b, P2G_CAND[c], GRID_CAND[c], G2P_CAND[c], e, false, false);
            if (rc) return rc;
        }
    MPM_HIP(hipStreamSynchronize(b->stream));
    // median of the span [e[k0], e[k0 + 1]] over the rounds
    auto median = [&](size_t first, size_t stride, int k0, float &out) -> int {
        std::vector<float> t;
        for (int32_t r = 0; r < reps; ++r) {
            hipEvent_t *e = ev + (first + (size_t)r * stride) * per;
            float v = 0;
            MPM_HIP(hipEventElapsedTime(&v, e[k0], e[k0 + 1]));
            t.push_back(v);
        }
        std::sort(t.begin(), t.end());
        out = t[t.size() / 2];
        return MPM_OK;
    };
    float med[3][NCAND];
    for (int c = 0; c < NCAND; ++c)
        for (int j = 0; j < 3; ++j)
            if ((rc = median((size_t)c, NCAND, STAGE_BEGIN[j], med[j][c]))) return rc;
    int best[3] = {0, 0, 0};
    for (int j = 0; j < 3; ++j)
        for (int c = 1; c < NCAND; ++c)
            if (med[j][c] < med[j][best[j]]) best[j] = c;
    b->shape.p2g_workgroups = P2G_CAND[best[0]];
    b->shape.grid_workgroups = GRID_CAND[best[1]];
    b->shape.g2p_threads = G2P_CAND[best[2]];
    // values of p2g_tile with the chosen widths
    const size_t t0 = (size_t)reps * NCAND;
    for (int32_t r = 0; r < reps; ++r)
        for (int c = 0; c < NTILE; ++c) {
            hipEvent_t *e = ev + (t0 + (size_t)r * NTILE + c) * per;
            rc = one_step(b, b->shape.p2g_workgroups, b->shape.grid_workgroups, b->shape.g2p_threads, e, false, false);
            if (rc) return rc;
        }
    if ((rc = release(b))) return rc;
    MPM_HIP(hipStreamSynchronize(b->stream));
    float tmed[NTILE];
    int tbest = 0;
    for (int c = 0; c < NTILE; ++c) {
        if ((rc = median(t0 + (size_t)c, NTILE, 0, tmed[c]))) return rc;
        if (tmed[c] < tmed[tbest]) tbest = c;
    }
    b->shape.p2g_tile = TILE_CAND[tbest];
    if (ms_out) {
        for (int j = 0; j < 3; ++j)
            for (int c = 0; c < NCAND; ++c) ms_out[j * NCAND + c] = med[j][c];
        for (int c = 0; c < NTILE; ++c) ms_out[3 * NCAND + c] = tmed[c];
    }
    return MPM_OK;
}

int mpm_batch_synchronize(mpm_batch *b)
{
    if (!b) return set_error(MPM_ERR_INVALID, "batch is null");
    MPM_HIP(hipStreamSynchronize(b->stream));
    return MPM_OK;
}

void mpm_batch_destroy(mpm_batch *b)
{
    if (!b) return;
    for (Chain &c : b->chains)
        if (c.stream) (void)hipStreamSynchronize(c.stream);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    drop_graphs(b);
    for (int p = 0; p < 2; ++p) {
        if (b->tab[p]) (void)hipFree(b->tab[p]);
        if (b->stab[p]) (void)hipFree(b->stab[p]);
    }
    if (b->ev_done) (void)hipEventDestroy(b->ev_done);
    if (b->ev_fork) (void)hipEventDestroy(b->ev_fork);
    for (Chain &c : b->chains) {
        if (c.stream) (void)hipStreamDestroy(c.stream);
        if (c.done) (void)hipEventDestroy(c.done);
    }
    for (hipEvent_t e : b->ev_join)
        if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : b->tev)
        if (e) (void)hipEventDestroy(e);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
}

}  // extern "C"
