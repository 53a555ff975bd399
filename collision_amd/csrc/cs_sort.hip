// Stable sort of (key, value) pairs for gfx950: up to RANK_SORT_MAX pairs by
// counting ranks, beyond that LSD radix passes.
//
// One radix pass per 8-bit digit, three kernels per pass (reduce-then-scan):
//   1. k_digit_hist  : per-tile 256-bin histogram (LDS atomics), written
//                      digit-major so a plain exclusive scan gives offsets.
//   2. exclusive_scan_u32 : device-wide scan of the histogram table.
//   3. k_scatter     : per-tile stable ranking.  Each 64-lane wavefront owns a
//                      contiguous quarter of the tile and walks it in 64-key
//                      rounds; lanes holding the same digit are found with 8
//                      ballots (one per digit bit), their rank is the popcount
//                      of lower matching lanes, and a per-wave LDS counter
//                      carries counts across rounds.  Keys keep their input
//                      order within a digit, so the sort is stable.
#include "cs_internal.h"

namespace cs {

constexpr int SORT_THREADS = 256;  // 4 wavefronts
constexpr int SORT_WAVES = SORT_THREADS / 64;
constexpr int SORT_ROUNDS = 8;     // keys per lane
constexpr int SORT_TILE = SORT_THREADS * SORT_ROUNDS;  // 2048
constexpr int SORT_SUB = SORT_TILE / SORT_WAVES;       // 512 keys per wave

template <typename K>
__global__ void __launch_bounds__(SORT_THREADS) k_digit_hist(const K* __restrict__ keys, int n,
                                                             int shift, uint32_t* __restrict__ hist,
                                                             int nblocks) {
  __shared__ uint32_t h[256];
  for (int i = threadIdx.x; i < 256; i += SORT_THREADS) h[i] = 0;
  __syncthreads();
  const int base = blockIdx.x * SORT_TILE;
  for (int k = threadIdx.x; k < SORT_TILE; k += SORT_THREADS) {
    int idx = base + k;
    if (idx < n) {
      uint32_t d = (uint32_t)((keys[idx] >> shift) & 255u);
      atomicAdd(&h[d], 1u);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 256; i += SORT_THREADS) hist[(size_t)i * nblocks + blockIdx.x] = h[i];
}

// Device-wide exclusive scan of uint32 in three coalesced phases:
// per-tile sums, one work-group scanning the tile sums, per-tile scan + offset.
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__global__ void __launch_bounds__(SCAN_THREADS) k_scan_reduce(const uint32_t* __restrict__ data,
                                                              int n, uint32_t* __restrict__ part) {
  __shared__ uint32_t red[SCAN_THREADS];
  const int base = blockIdx.x * SCAN_TILE;
  uint32_t s = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const int idx = base + k * SCAN_THREADS + threadIdx.x;
    if (idx < n) s += data[idx];
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int off = SCAN_THREADS / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// exclusive scan of part[0..np) by one work-group, in coalesced 1024-wide tiles
__global__ void __launch_bounds__(1024) k_scan_partials(uint32_t* __restrict__ part, int np) {
  __shared__ uint32_t buf[1024];
  __shared__ uint32_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int base = 0; base < np; base += 1024) {
    const int idx = base + threadIdx.x;
    const uint32_t v = idx < np ? part[idx] : 0u;
    buf[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      const uint32_t add = ((int)threadIdx.x >= off) ? buf[threadIdx.x - off] : 0u;
      __syncthreads();
      buf[threadIdx.x] += add;
      __syncthreads();
    }
    const uint32_t incl = buf[threadIdx.x];
    const uint32_t c = carry;
    if (idx < np) part[idx] = c + incl - v;
    __syncthreads();
    if (threadIdx.x == 1023) carry = c + incl;
    __syncthreads();
  }
}

__global__ void __launch_bounds__(SCAN_THREADS) k_scan_down(uint32_t* __restrict__ data, int n,
                                                            const uint32_t* __restrict__ part) {
  __shared__ uint32_t tile[SCAN_TILE];
  __shared__ uint32_t tsum[SCAN_THREADS];
  const int base = blockIdx.x * SCAN_TILE;
  const int t = threadIdx.x;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const int idx = base + k * SCAN_THREADS + t;
    tile[k * SCAN_THREADS + t] = idx < n ? data[idx] : 0u;
  }
  __syncthreads();
  uint32_t loc[SCAN_ITEMS];
  uint32_t run = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    loc[k] = run;
    run += tile[t * SCAN_ITEMS + k];
  }
  tsum[t] = run;
  __syncthreads();
  for (int off = 1; off < SCAN_THREADS; off <<= 1) {
    const uint32_t add = (t >= off) ? tsum[t - off] : 0u;
    __syncthreads();
    tsum[t] += add;
    __syncthreads();
  }
  const uint32_t pre = part[blockIdx.x] + tsum[t] - run;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) tile[t * SCAN_ITEMS + k] = pre + loc[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const int idx = base + k * SCAN_THREADS + t;
    if (idx < n) data[idx] = tile[k * SCAN_THREADS + t];
  }
}

size_t scan_partial_words(int n) { return (size_t)((n + SCAN_TILE - 1) / SCAN_TILE) + 1; }

hipError_t exclusive_scan_u32(hipStream_t st, uint32_t* data, int n, uint32_t* partials) {
  if (n <= 0) return hipSuccess;
  const int nt = (n + SCAN_TILE - 1) / SCAN_TILE;
  hipLaunchKernelGGL(k_scan_reduce, dim3(nt), dim3(SCAN_THREADS), 0, st, data, n, partials);
  hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(1024), 0, st, partials, nt);
  hipLaunchKernelGGL(k_scan_down, dim3(nt), dim3(SCAN_THREADS), 0, st, data, n, partials);
  return hipGetLastError();
}

template <typename K>
__global__ void __launch_bounds__(SORT_THREADS) k_scatter(const K* __restrict__ keys_in,
                                                          const uint32_t* __restrict__ vals_in,
                                                          K* __restrict__ keys_out,
                                                          uint32_t* __restrict__ vals_out, int n,
                                                          int shift,
                                                          const uint32_t* __restrict__ offsets,
                                                          int nblocks) {
  __shared__ uint32_t cnt[SORT_WAVES][256];
  __shared__ uint32_t boff[256];
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < SORT_WAVES * 256; i += SORT_THREADS) (&cnt[0][0])[i] = 0;
  for (int i = threadIdx.x; i < 256; i += SORT_THREADS)
    boff[i] = offsets[(size_t)i * nblocks + blockIdx.x];
  __syncthreads();

  const int base = blockIdx.x * SORT_TILE + w * SORT_SUB;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  K key[SORT_ROUNDS];
  uint32_t val[SORT_ROUNDS];
  uint32_t rank[SORT_ROUNDS];
  uint32_t dig[SORT_ROUNDS];
#pragma unroll
  for (int r = 0; r < SORT_ROUNDS; ++r) {
    const int idx = base + r * 64 + lane;
    const bool valid = idx < n;
    K k = valid ? keys_in[idx] : (K)0;
    uint32_t d = (uint32_t)((k >> shift) & 255u);
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      uint64_t bb = __ballot((d >> b) & 1u);
      peers &= ((d >> b) & 1u) ? bb : ~bb;
    }
    uint32_t before = cnt[w][d];
    if (valid) {
      const int leader = __ffsll((unsigned long long)peers) - 1;
      if (lane == leader) cnt[w][d] = before + (uint32_t)__popcll(peers);
    }
    rank[r] = before + (uint32_t)__popcll(peers & lt_mask);
    key[r] = k;
    val[r] = !valid ? 0u : vals_in ? vals_in[idx] : (uint32_t)idx;
    dig[r] = valid ? d : 256u;
  }
  __syncthreads();
  // exclusive prefix of the per-wave digit counts across the block's waves
  for (int d = threadIdx.x; d < 256; d += SORT_THREADS) {
    uint32_t run = 0;
#pragma unroll
    for (int ww = 0; ww < SORT_WAVES; ++ww) {
      uint32_t c = cnt[ww][d];
      cnt[ww][d] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < SORT_ROUNDS; ++r) {
    if (dig[r] < 256u) {
      const uint32_t pos = boff[dig[r]] + cnt[w][dig[r]] + rank[r];
      keys_out[pos] = key[r];
      vals_out[pos] = val[r];
    }
  }
}

// Small arrays (n <= RANK_SORT_MAX): a key's place in the stable order is the
// number of keys before it (smaller keys, and equal keys at smaller indices).
// A work-group places 64 keys, one per lane; its 16 wavefronts each count over a
// sixteenth of all keys, which are uniform across the wavefront and so come in
// through the scalar cache, eight per load: two instructions per comparison
// and no LDS traffic.  One launch, n / 64 work-groups.  It replaces a rank sort and
// an LDS radix sort in one work-group (800 64-bit keys 13.6 -> 3.8 us, 3,202 32-bit
// keys 20.7 -> 6 us) and, up to the limit, the radix passes' 5 launches per
// digit (32-bit keys, 4 digits: 7,938 keys 8 us against 100, 21,938 about 65 us
// against 20 launches of 4-8 us; the comparisons grow with the square).
constexpr int RANK_WAVES = 16;

// out(rank, i, key) is called once for each key i of the work-group
template <typename K, typename Out>
__device__ __attribute__((always_inline)) inline void rank_keys(const K* __restrict__ keys, int n,
                                                                Out out) {
  __shared__ int part[RANK_WAVES][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = blockIdx.x * 64, i = i0 + lane;
  const K ki = i < n ? keys[i] : (K)0;
  const int c0 = (int)((int64_t)n * w / RANK_WAVES), c1 = (int)((int64_t)n * (w + 1) / RANK_WAVES);
  int rank = 0;
  // [c0, c1) in three stretches: before this work-group's keys, among them, after
  auto count = [&](int a, int b, auto before) {
    int j = a;
    for (; j + 8 <= b; j += 8) {
      K k[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) k[u] = keys[j + u];
#pragma unroll
      for (int u = 0; u < 8; ++u) rank += before(k[u], j + u) ? 1 : 0;
    }
    for (; j < b; ++j) rank += before(keys[j], j) ? 1 : 0;
  };
  count(c0, min(c1, max(c0, i0)), [&](K k, int) { return k <= ki; });
  count(min(c1, max(c0, i0)), max(c0, min(c1, i0 + 64)),
        [&](K k, int j) { return k < ki || (k == ki && j < i); });
  count(max(c0, min(c1, i0 + 64)), c1, [&](K k, int) { return k < ki; });
  part[w][lane] = rank;
  __syncthreads();
  if (w == 0 && i < n) {
    int r = 0;
#pragma unroll
    for (int q = 0; q < RANK_WAVES; ++q) r += part[q][lane];
    out(r, i, ki);
  }
}

template <typename K>
__global__ void __launch_bounds__(64 * RANK_WAVES) k_sort_rank(const K* __restrict__ keys,
                                                              const uint32_t* __restrict__ vals,
                                                              K* __restrict__ keys_out,
                                                              uint32_t* __restrict__ vals_out, int n) {
  rank_keys(keys, n, [&](int r, int i, K k) {
    keys_out[r] = k;
    vals_out[r] = vals[i];
  });
}

// the hits in canonical order straight into their records: the sorted keys are
// not needed again (one launch instead of two, 2.3 us, at up to RANK_SORT_MAX hits)
__global__ void __launch_bounds__(64 * RANK_WAVES) k_rank_hits(const uint64_t* __restrict__ keys,
                                                              const hit_rec* __restrict__ hits, int n,
                                                              int nv, int nbody,
                                                              uint32_t* __restrict__ rkey,
                                                              uint32_t* __restrict__ rval) {
  rank_keys(keys, n, [&](int r, int i, uint64_t) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      rkey[4 * (size_t)r + p] = hit_record_key(hits[i], p, nv, nbody);
      rval[4 * (size_t)r + p] = (uint32_t)i * 4u + (uint32_t)p;
    }
  });
}

hipError_t rank_hits(hipStream_t st, const uint64_t* keys, const hit_rec* hits, int n, int nv,
                     int nbody, uint32_t* rkey, uint32_t* rval) {
  hipLaunchKernelGGL(k_rank_hits, dim3((n + 63) / 64), dim3(64 * RANK_WAVES), 0, st, keys, hits, n,
                     nv, nbody, rkey, rval);
  return hipGetLastError();
}

template <typename K>
static hipError_t radix_sort_impl(hipStream_t st, K* keys, uint32_t* vals, K* tmp_keys,
                                  uint32_t* tmp_vals, uint32_t* hist, uint32_t* partials, int n,
                                  int bits, bool* result_in_tmp, bool iota = false) {
  *result_in_tmp = false;
  if (n <= 1 || bits <= 0) return hipSuccess;
  if (n <= RANK_SORT_MAX) {
    hipLaunchKernelGGL(k_sort_rank<K>, dim3((n + 63) / 64), dim3(64 * RANK_WAVES), 0, st, keys,
                       vals, tmp_keys, tmp_vals, n);
    *result_in_tmp = true;
    return hipGetLastError();
  }
  const int nblocks = (n + SORT_TILE - 1) / SORT_TILE;
  K* kin = keys;
  uint32_t* vin = vals;
  K* kout = tmp_keys;
  uint32_t* vout = tmp_vals;
  for (int shift = 0; shift < bits; shift += 8) {
    hipLaunchKernelGGL(k_digit_hist<K>, dim3(nblocks), dim3(SORT_THREADS), 0, st, kin, n, shift,
                       hist, nblocks);
    CS_HIP_RET(exclusive_scan_u32(st, hist, 256 * nblocks, partials));
    hipLaunchKernelGGL(k_scatter<K>, dim3(nblocks), dim3(SORT_THREADS), 0, st, kin,
                       iota && shift == 0 ? nullptr : vin, kout, vout, n, shift, hist, nblocks);
    K* tk = kin; kin = kout; kout = tk;
    uint32_t* tv = vin; vin = vout; vout = tv;
    *result_in_tmp = !*result_in_tmp;
  }
  return hipGetLastError();
}

size_t radix_hist_words(int n) {
  const int nblocks = (n + SORT_TILE - 1) / SORT_TILE;
  return (size_t)256 * (nblocks > 0 ? nblocks : 1);
}

hipError_t radix_sort_u32(hipStream_t st, uint32_t* keys, uint32_t* vals, uint32_t* tmp_keys,
                          uint32_t* tmp_vals, uint32_t* hist, uint32_t* partials, int n, int bits,
                          bool* result_in_tmp) {
  return radix_sort_impl<uint32_t>(st, keys, vals, tmp_keys, tmp_vals, hist, partials, n, bits,
                                   result_in_tmp);
}

hipError_t radix_sort_u64(hipStream_t st, uint64_t* keys, uint32_t* vals, uint64_t* tmp_keys,
                          uint32_t* tmp_vals, uint32_t* hist, uint32_t* partials, int n, int bits,
                          bool* result_in_tmp, bool iota) {
  return radix_sort_impl<uint64_t>(st, keys, vals, tmp_keys, tmp_vals, hist, partials, n, bits,
                                   result_in_tmp, iota);
}

}  // namespace cs
