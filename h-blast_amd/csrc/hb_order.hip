// hb_order.hip -- orders a batched pass's HSPs by (query, oid, s_off, q_off).
//
// The scan emits records in any order with the group's contexts and offsets.
// An LSD radix sort of their keys, 8 bits a pass and only over the bits that
// the batch's queries and database can set, gives the order; the records
// themselves move once, mapped to their query's contexts and offsets on the
// way.  The bound is the launches: 296,000 records of 48 queries (6 passes,
// 21 launches) take 0.2 ms, where their copy to a fresh vector, partition and
// sort on the host took 7 ms of a batched pass.
#include <hip/hip_runtime.h>

#include "hb_internal.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / HB_WAVE;
constexpr int kRounds = 16;                                 // of 64 keys per wavefront
constexpr uint32_t kWaveKeys = kRounds * HB_WAVE;           // consecutive keys
constexpr uint32_t kBlockKeys = kWaves * kWaveKeys;
constexpr int kDigits = 256;

// lo = s_off, q_off within the query; hi = query, oid
__device__ __forceinline__ uint64_t key_of(const hb_order_args &a, uint32_t i, bool hi)
{
    const hb_hsp h = a.in[i];
    const int4 m = a.ctx_map[h.context];
    if (hi) return (uint64_t)(uint32_t)m.x << a.oid_bits | h.oid;
    return (uint64_t)(uint32_t)h.s_off << a.q_bits | (uint32_t)(h.q_off - m.z);
}

__global__ __launch_bounds__(kThreads) void order_lo_kernel(hb_order_args a)
{
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= a.n) return;
    a.sort.key[0][i] = key_of(a, i, false);
    a.sort.idx[0][i] = i;
}

__global__ __launch_bounds__(kThreads) void order_hi_kernel(hb_order_args a)
{
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i < a.n) a.sort.key[a.sort.src][i] = key_of(a, a.sort.idx[a.sort.src][i], true);
}

// Keys of each digit in each block: counts[digit * blocks + block].
__global__ __launch_bounds__(kThreads) void sort_count_kernel(const uint64_t *key, uint32_t n,
                                                               int shift, uint32_t *counts)
{
    __shared__ uint32_t h[kDigits];
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t i0 = blockIdx.x * kBlockKeys;
    for (uint32_t j = threadIdx.x; j < kBlockKeys; j += kThreads)
        if (i0 + j < n) atomicAdd(&h[(key[i0 + j] >> shift) & (kDigits - 1)], 1u);
    __syncthreads();
    counts[threadIdx.x * gridDim.x + blockIdx.x] = h[threadIdx.x];
}

__device__ __forceinline__ uint32_t block_excl(uint32_t v, uint32_t *sm, uint32_t *total)
{
    const int t = threadIdx.x;
    __syncthreads();
    sm[t] = v;
    __syncthreads();
    for (int o = 1; o < kThreads; o <<= 1) {
        const uint32_t x = t >= o ? sm[t - o] : 0u;
        __syncthreads();
        sm[t] += x;
        __syncthreads();
    }
    *total = sm[kThreads - 1];
    return sm[t] - v;
}

// One block per digit: its blocks' counts become exclusive sums, their total
// goes to totals[digit].
__global__ __launch_bounds__(kThreads) void sort_scan_kernel(uint32_t *counts, uint32_t blocks,
                                                              uint32_t *totals)
{
    __shared__ uint32_t sm[kThreads];
    uint32_t *c = counts + (size_t)blockIdx.x * blocks;
    uint32_t run = 0;
    for (uint32_t b0 = 0; b0 < blocks; b0 += kThreads) {
        const uint32_t b = b0 + threadIdx.x;
        uint32_t total;
        const uint32_t e = block_excl(b < blocks ? c[b] : 0u, sm, &total);
        if (b < blocks) c[b] = run + e;
        run += total;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = run;
}

// Moves keys and indices to their digit's place, in order: a wavefront takes
// kWaveKeys consecutive keys, 64 a round, and a key's rank among its digit's
// keys of the round is the number of lower lanes with the same digit.
__global__ __launch_bounds__(kThreads) void sort_move_kernel(const uint64_t *key,
                                                              const uint32_t *idx, uint32_t n,
                                                              int shift, const uint32_t *counts,
                                                              const uint32_t *totals,
                                                              uint64_t *key_out, uint32_t *idx_out)
{
    __shared__ uint32_t sm[kThreads];
    __shared__ uint32_t cur[kWaves][kDigits];
    const int lane = threadIdx.x & (HB_WAVE - 1), wid = threadIdx.x / HB_WAVE;
    uint32_t total;
    const uint32_t base = block_excl(totals[threadIdx.x], sm, &total) +
                          counts[threadIdx.x * gridDim.x + blockIdx.x];
    for (int w = 0; w < kWaves; ++w) cur[w][threadIdx.x] = 0;
    __syncthreads();
    const uint32_t i0 = blockIdx.x * kBlockKeys + (uint32_t)wid * kWaveKeys + (uint32_t)lane;
    for (int r = 0; r < kRounds; ++r) {
        const uint32_t i = i0 + (uint32_t)(r * HB_WAVE);
        if (i < n) atomicAdd(&cur[wid][(key[i] >> shift) & (kDigits - 1)], 1u);
    }
    __syncthreads();
    uint32_t at = base;   // thread = digit: where each wavefront's keys of it start
    for (int w = 0; w < kWaves; ++w) {
        const uint32_t c = cur[w][threadIdx.x];
        cur[w][threadIdx.x] = at;
        at += c;
    }
    __syncthreads();
    for (int r = 0; r < kRounds; ++r) {
        const uint32_t i = i0 + (uint32_t)(r * HB_WAVE);
        const bool v = i < n;
        const uint64_t k = v ? key[i] : 0;
        const uint32_t d = (uint32_t)(k >> shift) & (kDigits - 1);
        uint64_t same = __builtin_amdgcn_ballot_w64(v);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t m = __builtin_amdgcn_ballot_w64((d >> b) & 1u);
            same &= (d >> b) & 1u ? m : ~m;
        }
        const uint32_t rank = __builtin_amdgcn_mbcnt_hi(
            (uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
        const uint32_t to = cur[wid][d] + rank;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (v) {
            key_out[to] = k;
            idx_out[to] = idx[i];
            if (rank == 0) cur[wid][d] = to + (uint32_t)__popcll(same);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// The records in order, with their query's contexts and offsets, and each
// query's first record (q_first[n_queries] = n).
__global__ __launch_bounds__(kThreads) void order_emit_kernel(hb_order_args a)
{
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= a.n) return;
    const uint32_t *idx = a.sort.idx[a.sort.src];
    hb_hsp h = a.in[idx[i]];
    const int4 m = a.ctx_map[h.context];
    int32_t prev = -1;
    if (i > 0) prev = a.ctx_map[a.in[idx[i - 1]].context].x;
    for (int32_t q = prev + 1; q <= m.x; ++q) a.q_first[q] = i;
    if (i == a.n - 1)
        for (int32_t q = m.x + 1; q <= a.n_queries; ++q) a.q_first[q] = a.n;
    h.context = m.y;
    h.q_start -= m.z;
    h.q_off -= m.z;
    a.out[i] = h;
}

}  // namespace

size_t hb_sort_scratch(uint32_t n)
{
    const size_t blocks = (n + kBlockKeys - 1) / kBlockKeys;
    const size_t b = (size_t)n * 2 * (sizeof(uint64_t) + sizeof(uint32_t)) +
                     (blocks + 1) * kDigits * sizeof(uint32_t);
    return (b + 15) & ~(size_t)15;
}

void hb_sort_init(hb_sort *s, uint32_t n, void *scratch)
{
    const uint32_t blocks = (n + kBlockKeys - 1) / kBlockKeys;
    s->n = n;
    s->src = 0;
    s->key[0] = static_cast<uint64_t *>(scratch);
    s->key[1] = s->key[0] + n;
    s->idx[0] = reinterpret_cast<uint32_t *>(s->key[1] + n);
    s->idx[1] = s->idx[0] + n;
    s->counts = s->idx[1] + n;
    s->totals = s->counts + (size_t)blocks * kDigits;
}

void hb_launch_sort(hb_sort *s, int bits, hipStream_t st)
{
    const uint32_t blocks = (s->n + kBlockKeys - 1) / kBlockKeys;
    for (int shift = 0; shift < bits; shift += 8, s->src ^= 1) {
        const int i = s->src, o = i ^ 1;
        hipLaunchKernelGGL(sort_count_kernel, dim3(blocks), dim3(kThreads), 0, st, s->key[i], s->n,
                           shift, s->counts);
        hipLaunchKernelGGL(sort_scan_kernel, dim3(kDigits), dim3(kThreads), 0, st, s->counts,
                           blocks, s->totals);
        hipLaunchKernelGGL(sort_move_kernel, dim3(blocks), dim3(kThreads), 0, st, s->key[i],
                           s->idx[i], s->n, shift, s->counts, s->totals, s->key[o], s->idx[o]);
    }
}

hipError_t hb_launch_order(hb_order_args a, void *scratch, hipStream_t st)
{
    if (a.n == 0) return hipSuccess;
    const uint32_t grid = (a.n + kThreads - 1) / kThreads;
    hb_sort_init(&a.sort, a.n, scratch);
    hipLaunchKernelGGL(order_lo_kernel, dim3(grid), dim3(kThreads), 0, st, a);
    hb_launch_sort(&a.sort, a.s_bits + a.q_bits, st);
    hipLaunchKernelGGL(order_hi_kernel, dim3(grid), dim3(kThreads), 0, st, a);
    hb_launch_sort(&a.sort, a.query_bits + a.oid_bits, st);
    hipLaunchKernelGGL(order_emit_kernel, dim3(grid), dim3(kThreads), 0, st, a);
    return hipGetLastError();
}
