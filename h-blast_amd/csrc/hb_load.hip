// hb_load.hip -- the scan's view of a database, made on the device from the
// packed residues and offsets: subject records in processing order
// (length-descending) and the copy of the residues in that order.
//
// The order is a stable radix sort of the lengths and the records' places a
// prefix sum of the padded lengths (bound by the launches: 80 us for 300,000
// subjects, behind the residues' upload; the host's sort and its upload took
// 2 ms).  The copy also checks every residue and pads the subjects' ends, so
// the residues are read once.  A block writes 16 KB of the copy, found by
// binary search in the records, 16 bytes a lane and 16 lanes a subject: 124 MB
// in 105 us (2.4 TB/s read and written) and 86 MB of a length-sorted volume
// in 50 us (3.4; a copy kernel reaches 3.5), where a byte per lane and a check
// and a clearing pass of their own took 320 and 200 us.
#include <hip/hip_runtime.h>

#include "hb_internal.h"

namespace {

constexpr int kThreads = 256;
constexpr uint32_t kItems = 16;                   // subjects of a thread in the prefix sum
constexpr uint32_t kSpan = kThreads * kItems;     // ... of a block
constexpr uint32_t kCopyBytes = 16384;            // of the copy, per block

__global__ __launch_bounds__(kThreads) void load_keys_kernel(hb_load_args a)
{
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= a.n) return;
    a.sort.key[0][i] = a.max_len - (a.offs[i + 1] - a.offs[i]);   // ascending: length descending
    a.sort.idx[0][i] = i;
}

__device__ __forceinline__ uint64_t block_excl(uint64_t v, uint64_t *sm, uint64_t *total)
{
    const int t = threadIdx.x;
    __syncthreads();
    sm[t] = v;
    __syncthreads();
    for (int o = 1; o < kThreads; o <<= 1) {
        const uint64_t x = t >= o ? sm[t - o] : 0;
        __syncthreads();
        sm[t] += x;
        __syncthreads();
    }
    *total = sm[kThreads - 1];
    return sm[t] - v;
}

// Padded bytes of the thread's subjects (in processing order).
__device__ __forceinline__ uint64_t thread_bytes(const hb_load_args &a, const uint64_t *key,
                                                 uint32_t i0)
{
    uint64_t s = 0;
    for (uint32_t k = 0; k < kItems; ++k)
        if (i0 + k < a.n) s += (a.max_len - key[i0 + k] + 15) & ~15ull;
    return s;
}

__global__ __launch_bounds__(kThreads) void load_sum_kernel(hb_load_args a, const uint64_t *key)
{
    __shared__ uint64_t sm[kThreads];
    uint64_t total;
    block_excl(thread_bytes(a, key, blockIdx.x * kSpan + threadIdx.x * kItems), sm, &total);
    if (threadIdx.x == 0) a.part[blockIdx.x] = total;
}

__global__ __launch_bounds__(kThreads) void load_part_kernel(uint64_t *part, uint32_t blocks)
{
    __shared__ uint64_t sm[kThreads];
    uint64_t run = 0;
    for (uint32_t b0 = 0; b0 < blocks; b0 += kThreads) {
        const uint32_t b = b0 + threadIdx.x;
        uint64_t total;
        const uint64_t e = block_excl(b < blocks ? part[b] : 0, sm, &total);
        if (b < blocks) part[b] = run + e;
        run += total;
    }
}

__global__ __launch_bounds__(kThreads) void load_records_kernel(hb_load_args a, const uint64_t *key,
                                                                const uint32_t *idx)
{
    __shared__ uint64_t sm[kThreads];
    const uint32_t i0 = blockIdx.x * kSpan + threadIdx.x * kItems;
    uint64_t total;
    uint64_t dst = a.part[blockIdx.x] + block_excl(thread_bytes(a, key, i0), sm, &total);
    for (uint32_t k = 0; k < kItems; ++k) {
        const uint32_t i = i0 + k;
        if (i >= a.n) break;
        const uint32_t len = (uint32_t)(a.max_len - key[i]);
        a.subj[i] = make_uint4(idx[i], len, (uint32_t)dst, (uint32_t)(dst >> 32));
        dst += (len + 15u) & ~15u;
    }
}

__device__ __forceinline__ uint64_t place(const uint4 &r) { return (uint64_t)r.z | (uint64_t)r.w << 32; }

// The residues carry 64 spare bytes, so a subject's last 16-byte load may
// pass its end.
__global__ __launch_bounds__(kThreads) void load_copy_kernel(hb_load_args a)
{
    const uint64_t b0 = (uint64_t)blockIdx.x * kCopyBytes, b1 = b0 + kCopyBytes;
    uint32_t lo = 0, hi = a.n;   // the last record placed at or before b0
    while (hi - lo > 1) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (place(a.subj[mid]) <= b0) lo = mid;
        else hi = mid;
    }
    uint32_t bad = 0;
    for (uint32_t s = lo + threadIdx.x / 16; s < a.n; s += kThreads / 16) {
        const uint4 r = a.subj[s];
        const uint64_t dst = place(r);
        if (dst >= b1) break;
        const uint8_t *src = a.res + a.offs[r.x];
        const uint64_t end = min(dst + ((r.y + 15u) & ~15u), b1);
        for (uint64_t c = max(dst, b0) + 16 * (threadIdx.x & 15u); c < end; c += 256) {
            const uint32_t j = (uint32_t)(c - dst);   // < r.y
            uint32_t v[4];
            __builtin_memcpy(v, src + j, 16);
            const uint32_t left = r.y - j;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                if (left < 4 * k + 4) v[k] = left > 4 * k ? v[k] & (0xffffffffu >> (8 * (4 * k + 4 - left))) : 0u;
                // some byte >= HB_ALPHA
                bad |= (((v[k] & 0x7f7f7f7fu) + (0x80u - HB_ALPHA) * 0x01010101u) | v[k]) & 0x80808080u;
            }
            *reinterpret_cast<uint4 *>(a.out + c) = make_uint4(v[0], v[1], v[2], v[3]);
        }
    }
    const uint64_t m = __builtin_amdgcn_ballot_w64(bad != 0);
    if (m && (threadIdx.x & (HB_WAVE - 1)) == (uint32_t)__builtin_ctzll(m)) atomicOr(a.flag, 1u);
}

}  // namespace

size_t hb_load_scratch(uint32_t n)
{
    return hb_sort_scratch(n) + ((size_t)n / kSpan + 1) * sizeof(uint64_t);
}

hipError_t hb_launch_load_records(hb_load_args a, void *scratch, hipStream_t st)
{
    if (a.n == 0) return hipSuccess;
    const uint32_t grid = (a.n + kThreads - 1) / kThreads, blocks = (a.n + kSpan - 1) / kSpan;
    hb_sort_init(&a.sort, a.n, scratch);
    a.part = reinterpret_cast<uint64_t *>(static_cast<char *>(scratch) + hb_sort_scratch(a.n));
    hipLaunchKernelGGL(load_keys_kernel, dim3(grid), dim3(kThreads), 0, st, a);
    hb_launch_sort(&a.sort, hb_bits_of(a.max_len), st);
    const uint64_t *key = a.sort.key[a.sort.src];
    hipLaunchKernelGGL(load_sum_kernel, dim3(blocks), dim3(kThreads), 0, st, a, key);
    hipLaunchKernelGGL(load_part_kernel, dim3(1), dim3(kThreads), 0, st, a.part, blocks);
    hipLaunchKernelGGL(load_records_kernel, dim3(blocks), dim3(kThreads), 0, st, a, key,
                       a.sort.idx[a.sort.src]);
    return hipGetLastError();
}

hipError_t hb_launch_load_copy(const hb_load_args &a, uint64_t bytes, hipStream_t st)
{
    if (a.n == 0 || bytes == 0) return hipSuccess;
    const uint64_t blocks = (bytes + kCopyBytes - 1) / kCopyBytes;
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    hipLaunchKernelGGL(load_copy_kernel, dim3((unsigned)blocks), dim3(kThreads), 0, st, a);
    return hipGetLastError();
}
