// Three-phase exclusive scan: per-block scans (1024 threads x 4 elements),
// a recursive scan of the block totals, then a uniform add per block.
#include "scan_u32.h"

namespace h2 {

namespace {

constexpr unsigned kThreads = 1024;
constexpr unsigned kPer = 4;
constexpr unsigned kTile = kThreads * kPer;

// `total`: where the whole sum goes when one block scans everything (null otherwise)
__global__ void __launch_bounds__(kThreads) scan_tile_kernel(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
    uint64_t n, uint32_t* __restrict__ block_sums, uint32_t* __restrict__ total)
{
    __shared__ uint32_t s[kThreads];
    const uint64_t base = (uint64_t)blockIdx.x * kTile + (uint64_t)threadIdx.x * kPer;
    uint32_t v[kPer];
    uint32_t sum = 0;
#pragma unroll
    for (unsigned k = 0; k < kPer; ++k) {
        v[k] = (base + k < n) ? in[base + k] : 0u;
        sum += v[k];
    }
    s[threadIdx.x] = sum;
    for (unsigned d = 1; d < kThreads; d <<= 1) {
        __syncthreads();
        uint32_t t = threadIdx.x >= d ? s[threadIdx.x - d] : 0u;
        __syncthreads();
        s[threadIdx.x] += t;
    }
    __syncthreads();
    uint32_t run = threadIdx.x ? s[threadIdx.x - 1] : 0u;
#pragma unroll
    for (unsigned k = 0; k < kPer; ++k) {
        if (base + k < n)
            out[base + k] = run;
        run += v[k];
    }
    if (threadIdx.x == kThreads - 1) {
        block_sums[blockIdx.x] = s[kThreads - 1];
        if (total)
            *total = s[kThreads - 1];
    }
}

// the last thread's element also gives the whole sum (`total`, if not null): its scanned value
// plus its input
__global__ void add_block_kernel(const uint32_t* __restrict__ in, uint32_t* __restrict__ out, uint64_t n,
    const uint32_t* __restrict__ block_pre, uint32_t* __restrict__ total)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const uint32_t v = out[i] + block_pre[i / kTile];
    out[i] = v;
    if (total && i == n - 1)
        *total = v + in[i];
}

} // namespace

uint64_t scan_u32_scratch(uint64_t n)
{
    uint64_t bytes = 0;
    while (n > 1) {
        uint64_t nb = (n + kTile - 1) / kTile;
        bytes += align_up(4 * (nb + 1), 256) * 2;
        n = nb;
    }
    return bytes + 256;
}

static RustError scan_rec(const uint32_t* in, uint32_t* out, uint64_t n, uint8_t* scratch, uint32_t* total,
    hipStream_t stream)
{
    const uint64_t nb = (n + kTile - 1) / kTile;
    uint32_t* sums = (uint32_t*)scratch;
    uint32_t* sums_pre = (uint32_t*)(scratch + align_up(4 * (nb + 1), 256));
    uint8_t* next = scratch + 2 * align_up(4 * (nb + 1), 256);
    scan_tile_kernel<<<(unsigned)nb, kThreads, 0, stream>>>(in, out, n, sums, nb == 1 ? total : nullptr);
    H2_LAUNCH_CHECK();
    if (nb > 1) {
        RustError e = scan_rec(sums, sums_pre, nb, next, nullptr, stream);
        if (e.code)
            return e;
        add_block_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(in, out, n, sums_pre, total);
        H2_LAUNCH_CHECK();
    }
    return ok();
}

RustError scan_u32_exclusive(const uint32_t* in, uint32_t* out, uint64_t n, void* scratch, hipStream_t stream)
{
    if (n == 0) {
        H2_TRY(hipMemsetAsync(out, 0, 4, stream));
        return ok();
    }
    return scan_rec(in, out, n, (uint8_t*)scratch, out + n, stream);
}

} // namespace h2
