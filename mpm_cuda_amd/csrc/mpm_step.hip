// mpm_step.hip -- HIP kernels of the explicit MPM step (gfx950).
//
// Reference: JerryYan97/MPM_CUDA src/simulator/MPMCUDA.cu -- P2G :310-433,
// VelUpdate :435-472, InterpolateAndMove :474-741, step :793-925.  Particles
// are FP32 structure-of-arrays; the grid is block-major (4^3 nodes per block)
// and only blocks touched by the current P2G are updated and read.
#include "mpm_g2p.h"
#include "mpm_launch.h"

#include <algorithm>

namespace mpm {

// ---------------------------------------------------------------------------
// Small utilities.
__global__ void k_zero_u32(uint32_t *p, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// ---------------------------------------------------------------------------
// PLAIN form P2G: one thread per particle, 27 nodes x 4 FP32 global atomics,
// the stress SVD evaluated here (MPMCUDA.cu:310-433).
template <int MAT>
__global__ void __launch_bounds__(256) k_p2g_atomic(GridP g, MatP mat, PartView pv, float dt,
                                                    int sweeps, int tau_stored, float4 *grid,
                                                    uint32_t *flags, uint32_t *counters)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= pv.n) return;
    dt = step_dt(g, dt);
    float x[3] = {ld(pv, PL_X, i), ld(pv, PL_X + 1, i), ld(pv, PL_X + 2, i)};
    Stencil s;
    uint32_t bits = make_stencil(g, x, s);
    Scatter sc;
    load_scatter<MAT>(pv, i, mat, dt, tau_stored != 0, sweeps, sc, counters);
#pragma unroll
    for (int ox = 0; ox < 3; ++ox)
#pragma unroll
        for (int oy = 0; oy < 3; ++oy)
#pragma unroll
            for (int oz = 0; oz < 3; ++oz) {
                float4 c = node_contrib(g, s, sc, ox, oy, oz);
                float *dst = (float *)(grid + node_slot(g, s.b[0] + ox, s.b[1] + oy, s.b[2] + oz));
                unsafeAtomicAdd(dst + 0, c.x);
                unsafeAtomicAdd(dst + 1, c.y);
                unsafeAtomicAdd(dst + 2, c.z);
                unsafeAtomicAdd(dst + 3, c.w);
            }
    mark_blocks(g, s.b, flags);
    if (bits) atomicOr(counters + CT_HEALTH, bits);
}

// ---------------------------------------------------------------------------
// Grid velocity update over active blocks (MPMCUDA.cu:435-472): v = p / m,
// gravity, walls.  One wave per active block.  Node (mass, momentum) is the sum of grid_mp (PLAIN-form scatter and
// FAST-form spills) and, in the FAST form, of the staged P2G arenas of the
// up to 2x2x2 particle blocks whose arenas cover the node.  grid_mp is
// cleared for the next step; the result goes to grid_v.
// A block of the list is updated when marked, its mark cleared and the step
// number `seq` put in its act entry.
// The staging slots are looked up GB groups at a time (1, or 4 where there are
// more groups).
template <int GB>
__device__ __forceinline__ void grid_block(const GridP &g, float dt, uint32_t b, uint32_t *flags, uint32_t *act,
                                           uint32_t seq, float4 *gmp, float4 *gv,
                                           const float4 *__restrict__ staging, const int32_t *__restrict__ blk_tile,
                                           int ngroups, uint32_t staging_cap, int64_t nblocks)
{
    const int lane = threadIdx.x & 63;
    const int kx = lane & 3, ky = (lane >> 2) & 3, kz = lane >> 4;
    const uint32_t row = div_by(b, (uint32_t)g.nbx, g.div_nbx);
    const int bz = (int)div_by(row, (uint32_t)g.nby, g.div_nby);
    const int bx = (int)(b - row * (uint32_t)g.nbx), by = (int)row - bz * g.nby;
    const int64_t idx = (int64_t)b * BLK_NODES + lane;
    // Lanes 0..26 look up the staging slots of the 27 neighbour blocks at
    // once; with the mark and the block's own sums these loads are all in
    // flight together.
    const int px = bx + lane % 3 - 1, py = by + (lane / 3) % 3 - 1, pz = bz + lane / 9 - 1;
    const bool near = blk_tile && lane < 27 && px >= 0 && py >= 0 && pz >= 0 && px < g.nbx && py < g.nby && pz < g.nbz;
    const int32_t *bt = blk_tile + (((int64_t)pz * g.nby + py) * g.nbx + px);
    int32_t look[GB];
    auto lookup = [&](int g0) {
#pragma unroll
        for (int k = 0; k < GB; ++k) look[k] = near && g0 + k < ngroups ? gp(bt)[(int64_t)(g0 + k) * nblocks] : -1;
    };
    lookup(0);
    float4 a = gload4(gmp, idx);
    const uint32_t f = (uint32_t)__builtin_amdgcn_readfirstlane((int)gp(flags)[b]);
    if (!(f & BF_MARKED)) return;
    if (lane == 0) {
        gp(flags)[b] = f & ~BF_MARKED;
        gp(act)[b] = seq;
    }
    if (a.x != 0.f || a.y != 0.f || a.z != 0.f || a.w != 0.f) gstore4(gmp, idx, make_float4(0.f, 0.f, 0.f, 0.f));
    if (blk_tile) {
        for (int g0 = 0; g0 < ngroups; g0 += GB) {
            if (g0) lookup(g0);
#pragma unroll 1
            for (int gk = 0; gk < GB && g0 + gk < ngroups; ++gk) {
            int32_t at = look[0];
#pragma unroll
            for (int k = 1; k < GB; ++k) at = gk == k ? look[k] : at;
            const int32_t my_t = at >= 0 && ((uint32_t)at & TILE_SLOT_MASK) < staging_cap ? at : -1;
            // A node lies in exactly 8 of the 27 arenas: per axis its own
            // block's (d = 0) and the one below (d = -1, local k <= 2) or
            // above (d = +1, k = 3).  A neighbour's arena is read at index 7
            // (k = 2, below) or 0 (k = 3, above) only when its P2G wrote that
            // face (tile_entry); index 0 and 7 hold zero otherwise, and are
            // not written.  All loads are issued before any is used.
            const int sx = kx == 3 ? 1 : -1, sy = ky == 3 ? 1 : -1, sz = kz == 3 ? 1 : -1;
            float4 v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int dx = (e & 1) ? sx : 0, dy = (e & 2) ? sy : 0, dz = (e & 4) ? sz : 0;
                const int32_t t = __shfl(my_t, (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1));
                const int ax = kx + 1 - 4 * dx, ay = ky + 1 - 4 * dy, az = kz + 1 - 4 * dz;
                const uint32_t f = (uint32_t)t >> TILE_FACE_SHIFT;
                const bool face_ok = (ax != 0 || (f & 1u)) && (ax != 7 || (f & 2u)) && (ay != 0 || (f & 4u)) &&
                                     (ay != 7 || (f & 8u)) && (az != 0 || (f & 16u)) && (az != 7 || (f & 32u));
                const bool use = t >= 0 && face_ok;
                const int64_t ts = use ? (int64_t)((uint32_t)t & TILE_SLOT_MASK) : 0;
                v[e] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (use) v[e] = gload4(staging, ts * ARENA_NODES + (az * ARENA + ay) * ARENA + ax);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) { a.x += v[e].x; a.y += v[e].y; a.z += v[e].z; a.w += v[e].w; }
            }
        }
    }
    float4 out = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!(fabsf(a.x) < 2.220446049250313e-16f)) {          // MPMCUDA.cu:444
        const int ix = bx * BLK + kx, iy = by * BLK + ky, iz = bz * BLK + kz;
        float vx = a.y / a.x + g.gx * dt;                  // MPMCUDA.cu:452-457
        float vy = a.z / a.x + g.gy * dt;
        float vz = a.w / a.x + g.gz * dt;
        bool wx = ix <= g.pad || ix >= g.nx - g.pad;       // MPMCUDA.cu:463-469
        bool wy = iy <= g.pad || iy >= g.ny - g.pad;
        bool wz = iz <= g.pad || iz >= g.nz - g.pad;
        if (g.bc_mode == MPM_BC_STICKY) {
            if (wx || wy || wz) vx = vy = vz = 0.f;
        } else {
            if (wx) vx = 0.f;
            if (wy) vy = 0.f;
            if (wz) vz = 0.f;
        }
        out = make_float4(vx, vy, vz, a.x);
    }
    gstore4(gv, idx, out);
}

// Persistent over the list.  Also moves the step's spill count to CT_SPILLED,
// clears CT_SPILL for the next P2G and, when host_count (pinned host memory)
// is given, writes the count there and then the tile launch number to
// host_seq (a release store: a host that reads its launch's number also reads
// that launch's count).
template <int GB>
__global__ void __launch_bounds__(64) k_grid_update(GridP g, float dt, const uint32_t *list, uint32_t *flags,
                                                    uint32_t *act, uint32_t seq, uint32_t *counters, float4 *gmp,
                                                    float4 *gv, const float4 *__restrict__ staging,
                                                    const int32_t *__restrict__ blk_tile, int ngroups,
                                                    uint32_t staging_cap, int64_t nblocks, uint32_t *host_count,
                                                    uint32_t *host_seq, uint32_t launch, int clear_maxima)
{
    if (clear_maxima && blockIdx.x == 0) {
        static_assert(CT_MAXIMA == 64, "one copy per thread");
        gp(counters)[CT_COUNT * (1 + (int)threadIdx.x) + CT_SPEED] = 0u;
        gp(counters)[CT_COUNT * (1 + (int)threadIdx.x) + CT_DEFORM] = 0u;
    }
    const uint32_t n = counters[CT_LIST], n8 = round_xcd(n);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const uint32_t spilled = gp(counters)[CT_SPILL];
        gp(counters)[CT_SPILLED] = spilled;
        gp(counters)[CT_SPILL] = 0u;
        if (host_count) {
            *host_count = spilled;
            __hip_atomic_store(host_seq, launch, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    dt = step_dt(g, dt);
    for (uint32_t k8 = blockIdx.x; k8 < n8; k8 += gridDim.x) {
        const uint32_t k = xcd_spread(k8, n8);
        if (k >= n) continue;
        const uint32_t b = (uint32_t)__builtin_amdgcn_readfirstlane((int)list[k]);
        grid_block<GB>(g, dt, b, flags, act, seq, gmp, gv, staging, blk_tile, ngroups, staging_cap, nblocks);
    }
}

// Lists 256 consecutive blocks (thread t: block b0 + t) that `want`, with one
// global atomic: wave counts are combined in LDS.
__device__ __forceinline__ void list_blocks(bool want, int b0, uint32_t *list, uint32_t *counters)
{
    __shared__ uint32_t wave_cnt[4], wg_base;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t mask = __ballot(want);
    if (lane == 0) wave_cnt[w] = (uint32_t)__popcll(mask);
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t tot = wave_cnt[0] + wave_cnt[1] + wave_cnt[2] + wave_cnt[3];
        wg_base = tot ? gatomic_add(counters + CT_LIST, tot) : 0u;
    }
    __syncthreads();
    uint32_t off = wg_base;
    for (int k = 0; k < w; ++k) off += wave_cnt[k];
    if (want) gp(list)[off + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = (uint32_t)(b0 + (int)threadIdx.x);
}

// The blocks that the P2G marked (PLAIN form, each step).
__global__ void __launch_bounds__(256) k_list_marked(const uint32_t *flags, int nblocks, uint32_t *list,
                                                     uint32_t *counters)
{
    const int b0 = (int)(blockIdx.x * 256u), b = b0 + (int)threadIdx.x;
    list_blocks(b < nblocks && (gp(flags)[b] & BF_MARKED), b0, list, counters);
}

// Every tile's block and the next one in each axis (at each sort; a list of
// the marked blocks was a launch of every step, 4.6 us of 42 for 100k
// particles), and the blocks still marked.
__device__ __forceinline__ void list_near_tiles(const GridP &g, const int32_t *__restrict__ blk_tile, int ngroups,
                                                int nblocks, int b0, uint32_t *flags, uint32_t *list,
                                                uint32_t *counters)
{
    const int b = b0 + (int)threadIdx.x;
    uint32_t f = 0;
    if (b < nblocks) {
        const uint32_t row = div_by((uint32_t)b, (uint32_t)g.nbx, g.div_nbx);
        const int bz = (int)div_by(row, (uint32_t)g.nby, g.div_nby);
        const int bx = b - (int)row * g.nbx, by = (int)row - bz * g.nby;
        bool near = false;
        for (int gi = 0; gi < ngroups && !near; ++gi)
            for (int z = max(bz - 1, 0); z <= bz; ++z)
                for (int y = max(by - 1, 0); y <= by; ++y)
                    for (int x = max(bx - 1, 0); x <= bx; ++x)
                        near |= gp(blk_tile)[(int64_t)gi * nblocks + ((int64_t)z * g.nby + y) * g.nbx + x] >= 0;
        const uint32_t old = gp(flags)[b];
        f = (old & BF_MARKED) | (near || (old & BF_MARKED) ? BF_LISTED : 0u);
        if (f != old) gp(flags)[b] = f;
    }
    list_blocks(f != 0u, b0, list, counters);
}

__global__ void __launch_bounds__(256) k_list_near(GridP g, const int32_t *__restrict__ blk_tile, int ngroups,
                                                   int nblocks, uint32_t *flags, uint32_t *list, uint32_t *counters)
{
    list_near_tiles(g, blk_tile, ngroups, nblocks, (int)(blockIdx.x * 256u), flags, list, counters);
}

__global__ void __launch_bounds__(256) k_bsort_list(const SortSlice *__restrict__ tab, int ns)
{
    SliceScan sc;
    sc.build(ns, [&](int s) { return (uint32_t)((tab[s].nblocks + 255) / 256); });
    if (blockIdx.x >= sc.total) return;
    const uint32_t sid = (uint32_t)__builtin_amdgcn_readfirstlane((int)sc.find(blockIdx.x));
    const SortSlice &t = tab[sid];
    list_near_tiles(t.g, t.blk_tile, 1, t.nblocks, (int)((blockIdx.x - sc.start(sid)) * 256u), t.flags, t.list,
                    t.counters);
}

// Blocks whose act entry is `seq` (BATCH_SEQ: the device's own count of a
// batched scene) into CT_ACTIVE and, with gv, their nodes with mass into
// CT_NODES (statistics only).  One atomic per workgroup: same-address atomics
// from every wave would serialize in L2.
__global__ void __launch_bounds__(256) k_count_active(const uint32_t *act, uint32_t seq, int64_t nblocks,
                                                      uint32_t *counters, const float4 *__restrict__ gv)
{
    __shared__ uint32_t part[2][4];
    if (seq == BATCH_SEQ) seq |= counters[CT_SEQ];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t blocks = 0, nodes = 0;
    for (int64_t b0 = ((int64_t)blockIdx.x * 4 + w) * 64; b0 < nblocks; b0 += (int64_t)gridDim.x * 256) {
        const uint64_t m = __ballot(b0 + lane < nblocks && act[b0 + lane] == seq);
        blocks += (uint32_t)__popcll(m);
        if (gv)
            for (uint64_t r = m; r; r &= r - 1) {
                const float4 v = gv[(b0 + __ffsll((unsigned long long)r) - 1) * BLK_NODES + lane];
                nodes += (uint32_t)__popcll(__ballot(v.w != 0.f));
            }
    }
    if (lane == 0) {
        part[0][w] = blocks;
        part[1][w] = nodes;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        const uint32_t *p = part[threadIdx.x];
        const uint32_t t = p[0] + p[1] + p[2] + p[3];
        if (t) atomicAdd(counters + (threadIdx.x ? CT_NODES : CT_ACTIVE), t);
    }
}

int launch_count_active(hipStream_t st, const uint32_t *act, uint32_t seq, int64_t nblocks, uint32_t *counters,
                        const float4 *gv)
{
    if (int rc = launch_zero_u32(st, counters + CT_ACTIVE, 1)) return rc;
    if (gv)
        if (int rc = launch_zero_u32(st, counters + CT_NODES, 1)) return rc;
    hipLaunchKernelGGL(k_count_active, dim3(256), dim3(256), 0, st, act, seq, nblocks, counters, gv);
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// G2P, deformation update and advection, one thread per particle
// (MPMCUDA.cu:474-741).  With write_tau the Kirchhoff stress of the updated
// state is stored for the next P2G, so a FAST-form step needs one SVD.
// With sd, the step-size controller's measures of the updated particle are
// returned in sd[0] (speed) and sd[1] (deformation).
// Particle i of pv goes to slot io of po (see g2p_core).
template <int MAT>
__device__ __forceinline__ void g2p_particle(const GridP &g, const MatP &mat, const PartView &pv, int i,
                                             const PartView &po, int io, float dt, const float4 *__restrict__ gv,
                                             bool write_tau, int sweeps, uint32_t *counters, float *sd = nullptr)
{
    G2POut o;
    GlobalFetch f{gv};
    uint32_t bits = g2p_core<MAT>(g, mat, pv, i, po, io, dt, f, write_tau && MAT != MPM_WATER, sweeps, counters, o);
    if (write_tau && MAT != MPM_WATER) {
#pragma unroll
        for (int k = 0; k < 6; ++k) st(po, PL_TAU + k, io, o.tau[k]);
    }
    if (bits) gatomic_or(counters + CT_HEALTH, bits);
    if (sd) dt_measures<MAT>(mat, o.v, o.S, sd[0], sd[1]);
}

// Jello and snow G2P fit 128 VGPRs without spills when asked for four waves
// per SIMD (the default allocation took 131-133, three waves; 1M snow G2P
// 45.1 vs 47.0 us, measured); water's fits by default, and asking spilled.
template <int MAT>
constexpr int kG2pWaves = MAT == MPM_WATER ? 1 : 4;

// With the step-size controller on (g.dtp), every wave also merges its
// particles' maxima into counters[CT_SPEED], counters[CT_DEFORM] for the
// next step's control.  With a permutation (the re-sort of this step, FAST
// form) thread j updates particle perm[j] of pv into slot j of po (the other
// particle buffer), with its id and, when copy_q, its warm-start quaternion:
// the G2P itself moves the particles into their new order.
template <int MAT, bool MOVE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kG2pWaves<MAT>))) k_g2p(GridP g, MatP mat, PartView pv, float dt,
                                             const float4 *__restrict__ gv, int write_tau,
                                             int sweeps, uint32_t *counters, const uint32_t *__restrict__ perm,
                                             PartView po, const uint32_t *__restrict__ pid, uint32_t *pid_out,
                                             int copy_q)
{
    const uint32_t nb = ((uint32_t)pv.n + blockDim.x - 1) / blockDim.x;
    const uint32_t blk = xcd_spread(blockIdx.x, round_xcd(nb));      // launched with round_xcd(nb) workgroups
    if (blk >= nb) return;                                             // whole workgroup
    const int j = (int)(blk * blockDim.x + threadIdx.x);
    int i = j;
    if (MOVE && j < pv.n) {
        const uint32_t src = gp(perm)[j];
        i = src < (uint32_t)pv.n ? (int)src : j;     // always a valid index for a permutation
        gp(pid_out)[pv.off + j] = gp(pid)[pv.off + i];
        if (copy_q) {
#pragma unroll
            for (int k = 0; k < 4; ++k) st(po, PL_Q + k, j, ld(pv, PL_Q + k, i));
        }
    }
    const PartView &out = MOVE ? po : pv;        // chosen at compile time (one instantiation per case)
    if (!g.dtp) {
        if (j < pv.n) g2p_particle<MAT>(g, mat, pv, i, out, j, dt, gv, write_tau != 0, sweeps, counters);
        return;
    }
    dt = step_dt(g, dt);
    float sd[2] = {0.0f, 0.0f};
    if (j < pv.n) g2p_particle<MAT>(g, mat, pv, i, out, j, dt, gv, write_tau != 0, sweeps, counters, sd);
    wave_max_to(spread_maxima(counters) + CT_SPEED, sd[0]);
    wave_max_to(spread_maxima(counters) + CT_DEFORM, sd[1]);
}

// The FAST-form G2P of several groups in one launch, each group's particles in
// workgroups of their own: a launch costs 4.6 us, and 100k particles (12 us)
// fill no more than a wave a SIMD.  Jello, snow and water, 100k particles
// each: 8.9, 11.9 and 6.8 us apart, 17.4 together.
template <bool MOVE, bool CTL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_g2p_groups(const G2PArgs a)
{
    const uint32_t nb = a.grp[a.ngroups - 1].end, blk = xcd_spread(blockIdx.x, round_xcd(nb));
    if (blk >= nb) return;                                             // whole workgroup
    int gi = 0;
    while (a.grp[gi].end <= blk) ++gi;
    const G2PGroup &q = a.grp[gi];
    const int j = (int)((blk - (gi ? a.grp[gi - 1].end : 0u)) * blockDim.x + threadIdx.x);
    int i = j;
    PartView po = q.pv;
    if (MOVE) {
        po.P = q.P_out;
        if (j < q.pv.n) {
            const uint32_t src = gp(q.perm)[j];
            i = src < (uint32_t)q.pv.n ? (int)src : j;     // always a valid index for a permutation
            gp(a.pid_out)[q.pv.off + j] = gp(a.pid)[q.pv.off + i];
            if (a.copy_q) {
#pragma unroll
                for (int k = 0; k < 4; ++k) st(po, PL_Q + k, j, ld(q.pv, PL_Q + k, i));
            }
        }
    }
    const float dt = step_dt(a.g, a.dt);
    float sd[2] = {0.0f, 0.0f};
    float *measures = CTL ? sd : nullptr;
    if (j < q.pv.n) {
        switch (q.mat.type) {
        case MPM_JELLO: g2p_particle<MPM_JELLO>(a.g, q.mat, q.pv, i, po, j, dt, a.gv, true, a.sweeps, a.counters, measures); break;
        case MPM_SNOW: g2p_particle<MPM_SNOW>(a.g, q.mat, q.pv, i, po, j, dt, a.gv, true, a.sweeps, a.counters, measures); break;
        default: g2p_particle<MPM_WATER>(a.g, q.mat, q.pv, i, po, j, dt, a.gv, true, a.sweeps, a.counters, measures); break;
        }
    }
    if (!CTL) return;
    wave_max_to(spread_maxima(a.counters) + CT_SPEED, sd[0]);
    wave_max_to(spread_maxima(a.counters) + CT_DEFORM, sd[1]);
}

int launch_g2p_groups(hipStream_t st, const G2PArgs &a, uint32_t wgs, int threads, bool move)
{
    const dim3 gr(round_xcd(wgs)), bl(threads);
    const auto k = a.g.dtp ? (move ? k_g2p_groups<true, true> : k_g2p_groups<false, true>)
                           : (move ? k_g2p_groups<true, false> : k_g2p_groups<false, false>);
    hipLaunchKernelGGL(k, gr, bl, 0, st, a);
    return (int)hipGetLastError();
}

// FUSED form: the particles a tile kernel listed, persistent over the list.
// host_count (pinned host memory) receives their number, then host_seq the
// tile launch number `seq` (a release store: a host that reads seq == its
// launch also reads that launch's count).
template <int MAT>
__global__ void __launch_bounds__(256) k_p2g_spill(GridP g, MatP mat, PartView pv, float dt,
                                                   const uint32_t *__restrict__ list, uint32_t *counters,
                                                   float4 *grid, uint32_t *flags, uint32_t *blocks, uint32_t list_cap,
                                                   uint32_t *host_count, uint32_t *host_seq, uint32_t seq)
{
    const uint32_t listed = counters[CT_SPILL];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *host_count = listed;
        __hip_atomic_store(host_seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    const uint32_t n = min(listed, list_cap);
    dt = step_dt(g, dt);
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const int i = (int)list[k];
        if (i < 0 || i >= pv.n) continue;
        spill_particle<MAT>(g, mat, pv, i, dt, counters, grid, flags, blocks);
    }
}

// Kirchhoff stress of the current state, for the first P2G of the FAST form
// (and after the host rewrites F or J_p).
template <int MAT>
__global__ void k_compute_tau(MatP mat, PartView pv, int sweeps, uint32_t *counters)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= pv.n) return;
    float F[9], t[6];
#pragma unroll
    for (int k = 0; k < 9; ++k) F[k] = ld(pv, PL_F + k, i);
    float Jp = (MAT == MPM_SNOW) ? ld(pv, PL_S, i) : 1.0f;
    stress_from_F<MAT>(mat, F, Jp, sweeps, t, counters);
#pragma unroll
    for (int k = 0; k < 6; ++k) st(pv, PL_TAU + k, i, t[k]);
}

// ---------------------------------------------------------------------------
// Batched kernels: the scenes of a batch (BatchSlice table in device memory,
// one particle group per scene) in one launch per stage.  A workgroup maps
// its work index to a scene through a SliceScan of the per-scene counts,
// reads that scene's parameters with uniform loads and runs the body of the
// single-scene kernel.  Materials are selected per scene at run time.

// Grid update over the listed blocks of every scene (one wave per block).
// The first workgroup also does what k_grid_update does with the spill counts
// and hands the warm start's list over: the particles the last G2P listed go
// to this step's inference, and the list starts over for this step's G2P.
__global__ void __launch_bounds__(64) k_grid_batch(const BatchSlice *__restrict__ tab, int nslices)
{
    if (blockIdx.x == 0)
        for (int s = (int)threadIdx.x; s < nslices; s += 64) {
            const BatchSlice &b = tab[s];
            gp(b.counters)[CT_SPILLED] = gp(b.counters)[CT_SPILL];
            gp(b.counters)[CT_SPILL] = 0u;
            uint32_t *w = b.warm_cnt;
            if (w) {
                gp(w)[0] = gp(w)[1];
                gp(w)[1] = 0u;
            }
        }
    SliceScan sc;
    sc.build(nslices, [&](int s) { return gp(tab[s].counters)[CT_LIST]; });
    const uint32_t n = sc.total, n8 = round_xcd(n);
    for (uint32_t k8 = blockIdx.x; k8 < n8; k8 += gridDim.x) {
        const uint32_t k = xcd_spread(k8, n8);
        if (k >= n) continue;
        const uint32_t sid = (uint32_t)__builtin_amdgcn_readfirstlane((int)sc.find(k));
        const BatchSlice &b = tab[sid];
        const uint32_t blk = (uint32_t)__builtin_amdgcn_readfirstlane((int)gp(b.list)[k - sc.start(sid)]);
        grid_block<1>(b.g, b.dt, blk, b.flags, b.act, BATCH_SEQ | gp(b.counters)[CT_SEQ], b.grid_mp, b.grid_v, b.staging,
                    b.blk_tile, 1, b.staging_cap, b.nblocks);
    }
}

// G2P of every particle of the scenes (of material MATS, or of several:
// MAT_ANY); each scene's particles fill whole workgroups.  Launched with
// round_xcd(sum of ceil(n / blockDim)) workgroups.
template <int MATS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) k_g2p_batch(const BatchSlice *__restrict__ tab, int nslices)
{
    SliceScan sc;
    sc.build(nslices, [&](int s) { return ((uint32_t)tab[s].pv.n + blockDim.x - 1) / blockDim.x; });
    const uint32_t blk = xcd_spread(blockIdx.x, round_xcd(sc.total));
    if (blk >= sc.total) return;
    const uint32_t sid = (uint32_t)__builtin_amdgcn_readfirstlane((int)sc.find(blk));
    const BatchSlice &b = tab[sid];
    const int i = (int)((blk - sc.start(sid)) * blockDim.x + threadIdx.x);
    if (i >= b.pv.n) return;
    const int type = MATS == MAT_ANY ? b.mat.type : MATS;
    if (type == MPM_JELLO) g2p_particle<MPM_JELLO>(b.g, b.mat, b.pv, i, b.pv, i, b.dt, b.grid_v, true, b.sweeps, b.counters);
    else if (type == MPM_SNOW) g2p_particle<MPM_SNOW>(b.g, b.mat, b.pv, i, b.pv, i, b.dt, b.grid_v, true, b.sweeps, b.counters);
    else g2p_particle<MPM_WATER>(b.g, b.mat, b.pv, i, b.pv, i, b.dt, b.grid_v, true, b.sweeps, b.counters);
}

// A batch's re-sort move: every scene's particles from the buffers of table
// `src` into those of table `dst`, slot j taking particle perm[j] of the
// scene's last sort (all planes, the quaternions when copy_q, the ids); one
// thread per particle, each workgroup's 256 particles in one scene.
__global__ void __launch_bounds__(256) k_permute_batch(const BatchSlice *__restrict__ src,
                                                       const BatchSlice *__restrict__ dst, int nslices)
{
    SliceScan sc;
    sc.build(nslices, [&](int s) { return ((uint32_t)src[s].pv.n + 255u) / 256u; });
    const uint32_t blk = xcd_spread(blockIdx.x, round_xcd(sc.total));
    if (blk >= sc.total) return;
    const uint32_t sid = (uint32_t)__builtin_amdgcn_readfirstlane((int)sc.find(blk));
    const PartView a = src[sid].pv, b = dst[sid].pv;
    const int j = (int)((blk - sc.start(sid)) * 256u + threadIdx.x);
    if (j >= a.n) return;
    uint32_t from = gp(src[sid].perm)[j];
    if (from >= (uint32_t)a.n) from = (uint32_t)j;        // never taken for a valid permutation
    const bool q = src[sid].copy_q != 0;
    for (int p = 0; p < PL_COUNT; ++p)
        if (q || p < PL_Q || p >= PL_Q + 4) st(b, p, j, ld(a, p, (int)from));
    gp(b.pid)[b.off + j] = gp(a.pid)[a.off + (int64_t)from];
}

// ---------------------------------------------------------------------------
// Host-side launchers.
static inline int nblk(int64_t n, int t) { return (int)((n + t - 1) / t); }

int launch_zero_u32(hipStream_t st, uint32_t *p, int n)
{
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_zero_u32, dim3(nblk(n, 256)), dim3(256), 0, st, p, n);
    return (int)hipGetLastError();
}

int launch_p2g_atomic(hipStream_t st, const GridP &g, const MatP &m, const PartView &pv, float dt,
                      int sweeps, int tau_stored, float4 *grid, uint32_t *flags, uint32_t *counters,
                      int threads)
{
    if (pv.n <= 0) return 0;
    dim3 gr(nblk(pv.n, threads)), bl(threads);
    switch (m.type) {
    case MPM_JELLO: hipLaunchKernelGGL(k_p2g_atomic<MPM_JELLO>, gr, bl, 0, st, g, m, pv, dt, sweeps, tau_stored, grid, flags, counters); break;
    case MPM_SNOW: hipLaunchKernelGGL(k_p2g_atomic<MPM_SNOW>, gr, bl, 0, st, g, m, pv, dt, sweeps, tau_stored, grid, flags, counters); break;
    default: hipLaunchKernelGGL(k_p2g_atomic<MPM_WATER>, gr, bl, 0, st, g, m, pv, dt, sweeps, tau_stored, grid, flags, counters); break;
    }
    return (int)hipGetLastError();
}

int launch_list_marked(hipStream_t st, const uint32_t *flags, int nblocks, uint32_t *list, uint32_t *counters)
{
    if (int rc = launch_zero_u32(st, counters + CT_LIST, 1)) return rc;
    hipLaunchKernelGGL(k_list_marked, dim3(nblk(nblocks, 256)), dim3(256), 0, st, flags, nblocks, list, counters);
    return (int)hipGetLastError();
}

// CT_LIST was cleared (k_rank_tiles, k_bsort_rank).
int launch_list_near(hipStream_t st, const GridP &g, const int32_t *blk_tile, int ngroups, int nblocks, uint32_t *flags,
                     uint32_t *list, uint32_t *counters)
{
    hipLaunchKernelGGL(k_list_near, dim3(nblk(nblocks, 256)), dim3(256), 0, st, g, blk_tile, ngroups, nblocks, flags,
                       list, counters);
    return (int)hipGetLastError();
}

int launch_bsort_list(hipStream_t st, const SortSlice *tab, int ns, int wgs)
{
    hipLaunchKernelGGL(k_bsort_list, dim3(wgs), dim3(256), 0, st, tab, ns);
    return (int)hipGetLastError();
}

int launch_grid_update(hipStream_t st, const GridP &g, float dt, const uint32_t *list, uint32_t *flags, uint32_t *act,
                       uint32_t seq, uint32_t *counters, float4 *gmp, float4 *gv, int64_t nblocks,
                       const float4 *staging, const int32_t *blk_tile, int ngroups, uint32_t staging_cap,
                       uint32_t *host_count, uint32_t *host_seq, uint32_t launch, int clear_maxima)
{
    hipLaunchKernelGGL(ngroups > 1 ? k_grid_update<4> : k_grid_update<1>, dim3((uint32_t)std::min<int64_t>(nblocks, 8192)), dim3(64), 0, st, g, dt, list,
                       flags, act, seq, counters, gmp, gv, staging, blk_tile, ngroups, staging_cap, nblocks, host_count,
                       host_seq, launch, clear_maxima);
    return (int)hipGetLastError();
}

int launch_g2p(hipStream_t st, const GridP &g, const MatP &m, const PartView &pv, float dt,
               const float4 *gv, int write_tau, int sweeps, uint32_t *counters, int threads, const G2PMove *mv)
{
    if (pv.n <= 0) return 0;
    dim3 gr(round_xcd((uint32_t)nblk(pv.n, threads))), bl(threads);
    const G2PMove none{nullptr, pv, nullptr, nullptr, 0};
    const G2PMove &v = mv ? *mv : none;
    // the plain update and the one that moves particles are separate
    // instantiations: the move's index and buffer selection left the plain
    // kernel's registers and load schedule worse (G2P 41.2 vs 40.2 us median)
#define MPM_G2P_LAUNCH(MAT_)                                                                                    \
    do {                                                                                                        \
        if (mv) hipLaunchKernelGGL((k_g2p<MAT_, true>), gr, bl, 0, st, g, m, pv, dt, gv, write_tau, sweeps,     \
                                   counters, v.perm, v.po, v.pid, v.pid_out, v.copy_q);                         \
        else hipLaunchKernelGGL((k_g2p<MAT_, false>), gr, bl, 0, st, g, m, pv, dt, gv, write_tau, sweeps,       \
                                counters, v.perm, v.po, v.pid, v.pid_out, v.copy_q);                            \
    } while (0)
    switch (m.type) {
    case MPM_JELLO: MPM_G2P_LAUNCH(MPM_JELLO); break;
    case MPM_SNOW: MPM_G2P_LAUNCH(MPM_SNOW); break;
    default: MPM_G2P_LAUNCH(MPM_WATER); break;
    }
#undef MPM_G2P_LAUNCH
    return (int)hipGetLastError();
}

int launch_p2g_spill(hipStream_t st, const GridP &g, const MatP &m, const PartView &pv, float dt,
                     const uint32_t *list, uint32_t list_cap, uint32_t *counters, float4 *grid, uint32_t *flags, uint32_t *blocks,
                     uint32_t *host_count, uint32_t *host_seq, uint32_t seq)
{
    if (pv.n <= 0) return 0;
    if (!host_count || !host_seq) return (int)hipErrorInvalidValue;
    dim3 gr(64), bl(256);
    switch (m.type) {
    case MPM_JELLO: hipLaunchKernelGGL(k_p2g_spill<MPM_JELLO>, gr, bl, 0, st, g, m, pv, dt, list, counters, grid, flags, blocks, list_cap, host_count, host_seq, seq); break;
    case MPM_SNOW: hipLaunchKernelGGL(k_p2g_spill<MPM_SNOW>, gr, bl, 0, st, g, m, pv, dt, list, counters, grid, flags, blocks, list_cap, host_count, host_seq, seq); break;
    default: hipLaunchKernelGGL(k_p2g_spill<MPM_WATER>, gr, bl, 0, st, g, m, pv, dt, list, counters, grid, flags, blocks, list_cap, host_count, host_seq, seq); break;
    }
    return (int)hipGetLastError();
}

int launch_compute_tau(hipStream_t st, const MatP &m, const PartView &pv, int sweeps, uint32_t *counters)
{
    if (pv.n <= 0 || m.type == MPM_WATER) return 0;
    dim3 gr(nblk(pv.n, 256)), bl(256);
    if (m.type == MPM_JELLO)
        hipLaunchKernelGGL(k_compute_tau<MPM_JELLO>, gr, bl, 0, st, m, pv, sweeps, counters);
    else
        hipLaunchKernelGGL(k_compute_tau<MPM_SNOW>, gr, bl, 0, st, m, pv, sweeps, counters);
    return (int)hipGetLastError();
}

int launch_permute_batch(hipStream_t st, const BatchSlice *src, const BatchSlice *dst, int nslices, int wgs)
{
    if (wgs <= 0) return 0;
    hipLaunchKernelGGL(k_permute_batch, dim3(wgs), dim3(256), 0, st, src, dst, nslices);
    return (int)hipGetLastError();
}

int launch_grid_batch(hipStream_t st, const BatchSlice *tab, int nslices, int wgs)
{
    hipLaunchKernelGGL(k_grid_batch, dim3(wgs), dim3(64), 0, st, tab, nslices);
    return (int)hipGetLastError();
}

int launch_g2p_batch(hipStream_t st, int mats, const BatchSlice *tab, int nslices, int wgs, int threads)
{
    const auto kernel = mats == MPM_JELLO   ? k_g2p_batch<MPM_JELLO>
                        : mats == MPM_SNOW  ? k_g2p_batch<MPM_SNOW>
                        : mats == MPM_WATER ? k_g2p_batch<MPM_WATER>
                                            : k_g2p_batch<MAT_ANY>;
    hipLaunchKernelGGL(kernel, dim3(wgs), dim3(threads), 0, st, tab, nslices);
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// Step-size controller (no counterpart in the reference, which computes
// min(10, max_p max(J, 1/J)^3) after every step and never uses it,
// MPMCUDA.cu:915-920).  k_dt_scan reduces the controller's maxima over the
// current state (first step, or after the host rewrote particles); after
// that every G2P reduces them over the state it writes.  In the FAST form the
// P2G's waves turn the maxima into the step's dt themselves; in the PLAIN form
// k_dt_control does that first in each step, advances the clock and clears the
// maxima for this step's G2P.
template <int MAT>
__global__ void __launch_bounds__(256) k_dt_scan(MatP mat, PartView pv, uint32_t *counters)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    float sd[2] = {0.0f, 0.0f};
    if (i < pv.n) {
        const float v[3] = {ld(pv, PL_V, i), ld(pv, PL_V + 1, i), ld(pv, PL_V + 2, i)};
        float J;
        if (MAT == MPM_JELLO) {
            float F[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) F[k] = ld(pv, PL_F + k, i);
            J = det3<float>(F);
        } else {
            J = ld(pv, PL_S, i);
        }
        dt_measures<MAT>(mat, v, J, sd[0], sd[1]);
    }
    wave_max_to(spread_maxima(counters) + CT_SPEED, sd[0]);
    wave_max_to(spread_maxima(counters) + CT_DEFORM, sd[1]);
}

//
// The maxima are kept per workgroup copy of the counters: with one word each,
// the waves' atomics were two thirds of the G2P (100k particles of snow: 29
// us, 10.7 without the controller; now 13.6).
__global__ void __launch_bounds__(CT_SPREAD) k_dt_clear(uint32_t *counters)
{
    uint32_t *own = counters + CT_COUNT * (1 + threadIdx.x);
    gp(own)[CT_SPEED] = 0u;
    gp(own)[CT_DEFORM] = 0u;
}

__global__ void __launch_bounds__(CT_SPREAD) k_dt_control(DtRule rule, uint32_t *counters)
{
    __shared__ float part[2][CT_SPREAD / 64];
    uint32_t *own = counters + CT_COUNT * (1 + threadIdx.x);
    float speed = __uint_as_float(gp(own)[CT_SPEED]), deform = __uint_as_float(gp(own)[CT_DEFORM]);
    gp(own)[CT_SPEED] = 0u;
    gp(own)[CT_DEFORM] = 0u;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        speed = fmaxf(speed, __shfl_xor(speed, d));
        deform = fmaxf(deform, __shfl_xor(deform, d));
    }
    if ((threadIdx.x & 63) == 0) {
        part[0][threadIdx.x >> 6] = speed;
        part[1][threadIdx.x >> 6] = deform;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
#pragma unroll
    for (int w = 1; w < CT_SPREAD / 64; ++w) {
        speed = fmaxf(speed, part[0][w]);
        deform = fmaxf(deform, part[1][w]);
    }
    advance_clock(rule.ctl, control_dt(rule, speed, deform));
}

int launch_dt_clear(hipStream_t st, uint32_t *counters)
{
    hipLaunchKernelGGL(k_dt_clear, dim3(1), dim3(CT_SPREAD), 0, st, counters);
    return (int)hipGetLastError();
}

int launch_dt_scan(hipStream_t st, const MatP &m, const PartView &pv, uint32_t *counters)
{
    if (pv.n <= 0) return 0;
    dim3 gr(nblk(pv.n, 256)), bl(256);
    switch (m.type) {
    case MPM_JELLO: hipLaunchKernelGGL(k_dt_scan<MPM_JELLO>, gr, bl, 0, st, m, pv, counters); break;
    case MPM_SNOW: hipLaunchKernelGGL(k_dt_scan<MPM_SNOW>, gr, bl, 0, st, m, pv, counters); break;
    default: hipLaunchKernelGGL(k_dt_scan<MPM_WATER>, gr, bl, 0, st, m, pv, counters); break;
    }
    return (int)hipGetLastError();
}

int launch_dt_control(hipStream_t st, const DtRule &rule, uint32_t *counters)
{
    hipLaunchKernelGGL(k_dt_control, dim3(1), dim3(CT_SPREAD), 0, st, rule, counters);
    return (int)hipGetLastError();
}

}  // namespace mpm
