// mpm_read.hip -- particle fields to the host, in particle-id order.
//
// The reference copies its positions to the host after every step
// (MPMCUDA.cu:906-913); here particles are stored in planes in the order of
// the last block sort.  A read is one kernel that puts each
// particle's row in its place, and moves over the link only what the caller
// asked for.
#include "mpm_launch.h"

#include <algorithm>
#include <cstring>
#include <utility>

namespace mpm {

// Row i of W floats from the planes; `ids` gives each stored particle's row
// (NULL: its own index, offset j0).  Rows past n raise *bad instead.
template <int W>
__global__ void __launch_bounds__(256) k_read_rows(const float *__restrict__ planes, int64_t stride, int64_t j0,
                                                   int64_t m, uint32_t n, const uint32_t *__restrict__ ids,
                                                   float *__restrict__ out, uint32_t *bad)
{
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (j >= m) return;
    const uint32_t i = ids ? gp(ids)[j] : (uint32_t)j;
    if (i >= n) {
        *bad = 1u;
        return;
    }
    float v[W];
#pragma unroll
    for (int c = 0; c < W; ++c) v[c] = gp(planes)[c * stride + j0 + j];
    float *row = out + (int64_t)i * W;
#pragma unroll
    for (int c = 0; c < W; ++c) gp(row)[c] = v[c];
}

__global__ void __launch_bounds__(256) k_read_copy(const float4 *__restrict__ src, float4 *__restrict__ dst, int n)
{
    for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += gridDim.x * 256) gstore4(dst, k, gload4(src, k));
}

static void launch_rows(int w, hipStream_t st, const float *planes, int64_t stride, int64_t j0, int64_t m, int64_t n,
                        const uint32_t *ids, float *out, uint32_t *bad)
{
    const dim3 gr((unsigned)((m + 255) / 256)), bl(256);
    const uint32_t rows = (uint32_t)n;
    switch (w) {
    case 1: hipLaunchKernelGGL(k_read_rows<1>, gr, bl, 0, st, planes, stride, j0, m, rows, ids, out, bad); break;
    case 2: hipLaunchKernelGGL(k_read_rows<2>, gr, bl, 0, st, planes, stride, j0, m, rows, ids, out, bad); break;
    case 3: hipLaunchKernelGGL(k_read_rows<3>, gr, bl, 0, st, planes, stride, j0, m, rows, ids, out, bad); break;
    case 4: hipLaunchKernelGGL(k_read_rows<4>, gr, bl, 0, st, planes, stride, j0, m, rows, ids, out, bad); break;
    case 6: hipLaunchKernelGGL(k_read_rows<6>, gr, bl, 0, st, planes, stride, j0, m, rows, ids, out, bad); break;
    default: hipLaunchKernelGGL(k_read_rows<9>, gr, bl, 0, st, planes, stride, j0, m, rows, ids, out, bad); break;
    }
}

// Pinned buffers, READ_HEAD bytes (a flag word) and 64 KiB, 256 KiB, 1 MiB or
// READ_SLOTS slots: lent to one read at a time.  Allocating one costs ~0.2 ms,
// so up to POOL_KEEP stay for the next read of any simulator.
constexpr size_t READ_SLOT = (size_t)1 << 20, READ_HEAD = 64;
constexpr int POOL_KEEP = 4;
struct PinBuf {
    char *p;
    size_t size;
};
struct PinPool {
    std::mutex lock;
    PinBuf idle[POOL_KEEP];
    int count = 0;
    int users = 0;
};
static PinPool &pool()
{
    static PinPool *p = new PinPool();      // outlives static destructors
    return *p;
}

ReadStage::ReadStage()
{
    std::lock_guard<std::mutex> hold(pool().lock);
    pool().users += 1;
}

ReadStage::~ReadStage()
{
    for (hipEvent_t e : ev)
        if (e) (void)hipEventDestroy(e);
    std::lock_guard<std::mutex> hold(pool().lock);
    if (--pool().users) return;
    for (int k = 0; k < pool().count; ++k) (void)hipHostFree(pool().idle[k].p);
    pool().count = 0;
}

// A lent buffer, given back when the read ends (after the stream's work on it
// where the read ends early).
struct PinLoan {
    hipStream_t st;
    PinBuf b{nullptr, 0};
    bool settled = false;
    int take(size_t bytes)
    {
        {
            PinPool &q = pool();
            std::lock_guard<std::mutex> hold(q.lock);
            int best = -1;
            for (int k = 0; k < q.count; ++k)
                if (q.idle[k].size >= bytes && (best < 0 || q.idle[k].size < q.idle[best].size)) best = k;
            if (best >= 0) {
                b = q.idle[best];
                q.idle[best] = q.idle[--q.count];
                return MPM_OK;
            }
        }
        size_t size = (size_t)64 << 10;
        while (size < bytes) size *= 4;
        char *p = nullptr;
        MPM_HIP(hipHostMalloc((void **)&p, READ_HEAD + size, hipHostMallocPortable));
        b = PinBuf{p, size};
        return MPM_OK;
    }
    ~PinLoan()
    {
        if (!b.p) return;
        if (!settled) (void)hipStreamSynchronize(st);
        PinPool &q = pool();
        std::lock_guard<std::mutex> hold(q.lock);
        if (q.count == POOL_KEEP) {         // the smallest one goes
            int least = 0;
            for (int k = 1; k < POOL_KEEP; ++k)
                if (q.idle[k].size < q.idle[least].size) least = k;
            if (q.idle[least].size < b.size) std::swap(q.idle[least], b);
            (void)hipHostFree(b.p);
            return;
        }
        q.idle[q.count++] = b;
    }
};

// A read of up to READ_SLOT bytes: the kernel writes the rows straight to
// pinned memory (10k positions 14 us with the wait; through a device buffer
// and a copy 24, into pageable memory 71).  A larger one: rows in id order to
// `scratch`, then slot by slot over the link while the host copies the slots
// that arrived (2M positions: 24 MB at the link's 52 GB/s).
int read_rows(ReadStage &rs, hipStream_t st, const float *planes, int64_t stride, int64_t n, int w,
              const uint32_t *ids, float *scratch, float *out)
{
    if (n <= 0) {
        MPM_HIP(hipStreamSynchronize(st));
        return MPM_OK;
    }
    std::lock_guard<std::mutex> hold(rs.lock);
    const size_t bytes = (size_t)n * w * sizeof(float);
    const bool small = bytes <= READ_SLOT;
    PinLoan pin{st};
    int rc = pin.take(small ? bytes : READ_SLOT * READ_SLOTS);
    if (rc) return rc;
    uint32_t *const flag = (uint32_t *)pin.b.p;
    volatile uint32_t *bad = flag;
    char *const data = pin.b.p + READ_HEAD;
    *bad = 0u;
    const char *corrupt = "particle id table corrupted";
    if (small) {
        launch_rows(w, st, planes, stride, 0, n, n, ids, (float *)data, flag);
        MPM_HIP(hipGetLastError());
        MPM_HIP(hipStreamSynchronize(st));
        pin.settled = true;
        if (*bad) return set_error(MPM_ERR_STATE, corrupt);
        std::memcpy(out, data, bytes);
        return MPM_OK;
    }
    for (hipEvent_t &e : rs.ev)     // the rows are read by the host: release to the system
        if (!e) MPM_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventReleaseToSystem));
    if (ids) {
        launch_rows(w, st, planes, stride, 0, n, n, ids, scratch, flag);
        MPM_HIP(hipGetLastError());
    }
    // whole rows and whole 16 bytes a slot
    const int64_t per = (int64_t)(READ_SLOT / (16 * w)) * 4, slots = (n + per - 1) / per;
    auto send = [&](int64_t k) -> int {
        const int64_t j0 = k * per, m = std::min(per, n - j0);
        float *dst = (float *)(data + (k % READ_SLOTS) * READ_SLOT);
        if (ids)
            hipLaunchKernelGGL(k_read_copy, dim3(64), dim3(256), 0, st, (const float4 *)(scratch + j0 * w), (float4 *)dst,
                               (int)((m * w + 3) / 4));
        else
            launch_rows(w, st, planes, stride, j0, m, m, nullptr, dst, flag);
        MPM_HIP(hipGetLastError());
        MPM_HIP(hipEventRecord(rs.ev[k % READ_SLOTS], st));
        return MPM_OK;
    };
    for (int64_t k = 0; k < std::min<int64_t>(slots, READ_SLOTS) && !rc; ++k) rc = send(k);
    for (int64_t k = 0; k < slots && !rc; ++k) {
        MPM_HIP(hipEventSynchronize(rs.ev[k % READ_SLOTS]));
        const int64_t j0 = k * per, m = std::min(per, n - j0);
        std::memcpy(out + j0 * w, data + (k % READ_SLOTS) * READ_SLOT, (size_t)m * w * sizeof(float));
        if (k + READ_SLOTS < slots) rc = send(k + READ_SLOTS);
    }
    if (rc) return rc;
    MPM_HIP(hipStreamSynchronize(st));
    pin.settled = true;
    return *bad ? set_error(MPM_ERR_STATE, corrupt) : MPM_OK;
}

}  // namespace mpm
