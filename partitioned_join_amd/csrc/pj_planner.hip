// pj_planner.hip -- learned join planner for gfx950.
//
//   k_sketch          one workgroup: 4096 probe keys sampled at fixed strides,
//                     a 1024-bin histogram of their MurmurHash3 values (ordered
//                     by count, so the features describe the skew profile and
//                     not which bins it falls in), six size/skew scalars, and
//                     the 64 most frequent sampled keys as heavy candidates.
//   k_count_cand      exact occurrence counts of the candidates in the whole
//                     probe column (LDS hash of the candidates, one pass;
//                     16-byte vector loads when the column is aligned).
//   k_gemm, ...       a 1030 -> 256 -> 256 -> 81 FP32 MLP: forward, backward
//                     and Adam.  The products are tiny (batch <= a few hundred)
//                     so one LDS-tiled FP32 GEMM with strided operands serves
//                     the forward and both backward products.
// The planner only chooses the plan; the join result never depends on it.
#include <cmath>

#include "pj_device.h"
#include "pj_internal.h"
#include "pj_planner.h"

namespace pj {

// ---------------------------------------------------------------------------
// Sketch
// ---------------------------------------------------------------------------
// One workgroup, no sort of the sample: its distinct keys are counted in an
// LDS hash table (a slot holds the index of the sample that took it, so no key
// is reserved), bin counts are placed by counting (equal counts in any order
// give the same feature), and of the keys only the 64 candidates are ordered:
// those above the count that the 64th has, and the smallest keys of that
// count, found by a radix select.  Latency bounds it (a few waves of LDS work
// between barriers): 102 us with three bitonic sorts of up to 4096 values,
// 33 us here (16M x 256M Zipf(1.0)).
constexpr int kSketchSlots = 2 * kPlanSample;

// Exclusive prefix sums over r = 0 .. 4096 of s (r = 4096 last), in place, by
// 1024 threads.  Ends with a barrier.
__device__ __forceinline__ void scan_counts(uint32_t* s, uint32_t* s_tmp) {
  uint32_t v[4], sum = 0, total;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    v[c] = s[4 * threadIdx.x + c];
    sum += v[c];
  }
  uint32_t run = block_exclusive_scan<1024>(sum, s_tmp, &total);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    s[4 * threadIdx.x + c] = run;
    run += v[c];
  }
  if (threadIdx.x == 0) s[kPlanSample] = total;
  __syncthreads();
}

template <int KB>
__global__ __launch_bounds__(1024) void k_sketch(const void* keys, int64_t n, int64_t n_build, float* feat,
                                                 uint64_t* cand_keys, uint32_t* cand_counts) {
  using key_t = typename KeyT<KB>::key_t;
  __shared__ uint64_t s_key[kPlanSample];       // the sample
  __shared__ uint32_t s_cnt[kPlanSample];       // occurrences, at the sample index that owns the key's slot
  __shared__ uint32_t s_slot[kSketchSlots];     // owner + 1, 0: free; then the counts by count, below
  __shared__ uint32_t s_hist[kPlanBins];
  __shared__ uint32_t s_tmp[2][1024 / kWave + 1];
  __shared__ float s_red[1024 / kWave];
  __shared__ uint64_t s_ck[kPlanCand];
  __shared__ uint32_t s_cc[kPlanCand];
  __shared__ uint32_t s_sel[256], s_n, s_cstar, s_digit, s_left, s_top;
  const int tid = threadIdx.x;
  const key_t* k = static_cast<const key_t*>(keys);
  static_assert(kPlanSample == 4 * 1024 && kPlanBins == 1024, "four samples and one bin a thread");
  s_hist[tid] = 0;
#pragma unroll
  for (int c = 0; c < 4; ++c) s_cnt[4 * tid + c] = 0;
#pragma unroll
  for (int c = 0; c < kSketchSlots / 1024; ++c) s_slot[c * 1024 + tid] = 0;
  if (tid == 0) s_n = 0;
  uint64_t v[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int j = 4 * tid + c;
    v[c] = 0;
    if (n > 0) {
      const int64_t pos = ((2 * int64_t(j) + 1) * n) / (2 * int64_t(kPlanSample));  // < n
      v[c] = uint64_t(k[pos]);
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) s_key[4 * tid + c] = v[c];
  __syncthreads();
  if (n > 0) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t h = murmur3(key_t(v[c]));
      atomicAdd(&s_hist[h & uint32_t(kPlanBins - 1)], 1u);
      const uint32_t me = uint32_t(4 * tid + c);
      uint32_t s = (h >> 10) % uint32_t(kSketchSlots);
      while (true) {  // half the slots stay free
        const uint32_t o = atomicCAS(&s_slot[s], 0u, me + 1u);
        if (o == 0u || s_key[o - 1u] == v[c]) {
          atomicAdd(&s_cnt[o == 0u ? me : o - 1u], 1u);
          break;
        }
        s = (s + 1u) % uint32_t(kSketchSlots);
      }
    }
  }
  __syncthreads();
  // Distinct keys and bins by count, the largest first (r = 4096 - count).
  uint32_t* s_kr = s_slot;                      // [4097]
  __shared__ uint32_t s_br[kPlanSample + 1];
#pragma unroll
  for (int c = 0; c < 4; ++c) s_kr[c * 1024 + tid] = s_br[c * 1024 + tid] = 0;
  if (tid == 0) s_kr[kPlanSample] = s_br[kPlanSample] = 0;
  __syncthreads();
  float sq = 0.f;  // whole numbers up to 4096^2 = 2^24: exact in any order
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t cnt = s_cnt[4 * tid + c];
    sq += float(cnt) * float(cnt);
    if (cnt) atomicAdd(&s_kr[kPlanSample - cnt], 1u);
  }
  atomicAdd(&s_br[kPlanSample - s_hist[tid]], 1u);
  for (int d = kWave / 2; d > 0; d >>= 1) sq += __shfl_xor(sq, d, kWave);
  if ((tid & (kWave - 1)) == 0) s_red[tid / kWave] = sq;
  __syncthreads();
  scan_counts(s_kr, s_tmp[0]);
  scan_counts(s_br, s_tmp[1]);
  feat[atomicAdd(&s_br[kPlanSample - s_hist[tid]], 1u)] = float(s_hist[tid]) / float(kPlanSample);
  // The 64th key's count: r with fewer than 64 keys before it and 64 or more
  // up to it (fewer distinct keys than 64: the last r that has any).
  const uint32_t want = min(uint32_t(kPlanCand), s_kr[kPlanSample]);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t r = uint32_t(4 * tid + c), lo = s_kr[r], hi = s_kr[r + 1];
    if (lo < want && hi >= want) {
      s_cstar = uint32_t(kPlanSample) - r;
      s_left = want - lo;  // keys of that count to take
    }
    if (lo == 0 && hi > 0) s_top = uint32_t(kPlanSample) - r;
  }
  __syncthreads();
  // The s_left smallest of the keys with count cstar: their largest, digit by
  // digit from the top.
  uint64_t prefix = 0;
  if (want > 0) {
    const uint32_t cstar = s_cstar;
    for (int shift = KB * 8 - 8; shift >= 0; shift -= 8) {
      if (tid < 256) s_sel[tid] = 0;
      const uint32_t left = s_left;
      __syncthreads();
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (s_cnt[4 * tid + c] == cstar && (shift + 8 == KB * 8 || (v[c] >> (shift + 8)) == (prefix >> (shift + 8))))
          atomicAdd(&s_sel[uint32_t(v[c] >> shift) & 255u], 1u);
      __syncthreads();
      if (tid < kWave) {
        uint32_t q[4], sum = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          q[c] = s_sel[4 * tid + c];
          sum += q[c];
        }
        uint32_t run = sum;
        for (int d = 1; d < kWave; d <<= 1) {
          const uint32_t y = __shfl_up(run, d, kWave);
          if (tid >= d) run += y;
        }
        run -= sum;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if (run < left && run + q[c] >= left) {
            s_digit = uint32_t(4 * tid + c);
            s_left = left - run;
          }
          run += q[c];
        }
      }
      __syncthreads();
      prefix |= uint64_t(s_digit) << shift;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t cnt = s_cnt[4 * tid + c];
      if (cnt > cstar || (cnt == cstar && v[c] <= prefix)) {
        const uint32_t at = atomicAdd(&s_n, 1u);  // want of them: the keys are distinct
        if (at < uint32_t(kPlanCand)) {
          s_ck[at] = v[c];
          s_cc[at] = cnt;
        }
      }
    }
  }
  __syncthreads();
  if (tid < kPlanCand) {  // by count, then by key
    const uint32_t m = min(s_n, uint32_t(kPlanCand));
    if (uint32_t(tid) < m) {
      const uint64_t key = s_ck[tid];
      const uint32_t cnt = s_cc[tid];
      uint32_t rank = 0;
      for (uint32_t i = 0; i < m; ++i) rank += s_cc[i] > cnt || (s_cc[i] == cnt && s_ck[i] < key) ? 1u : 0u;
      cand_keys[rank] = key;
      cand_counts[rank] = cnt;
    } else {
      cand_keys[tid] = 0ull;
      cand_counts[tid] = 0u;
    }
  }
  if (tid == 0) {
    float tot = 0.f;
    for (int w = 0; w < 1024 / kWave; ++w) tot += s_red[w];
    const double nb = double(n_build) + 1.0, ns = double(n) + 1.0;
    feat[kPlanBins + 0] = float(log2(nb) / 32.0);
    feat[kPlanBins + 1] = float(log2(ns) / 32.0);
    feat[kPlanBins + 2] = float(log2(ns / nb) / 8.0);
    feat[kPlanBins + 3] = float(KB) / 8.0f;
    feat[kPlanBins + 4] = n > 0 ? float(s_top) / float(kPlanSample) : 0.f;
    feat[kPlanBins + 5] = n > 0 ? tot / (float(kPlanSample) * float(kPlanSample)) : 0.f;
  }
}

// ---------------------------------------------------------------------------
// Exact candidate counts: the valid candidates (sample count > 0) sit in a
// 128-slot LDS open-addressing table; every probe key is looked up once.  The
// table's slot is the top bits of a multiplicative hash (one multiply per
// key; the counts do not depend on it).
// ---------------------------------------------------------------------------
template <int SLOTS>
__device__ __forceinline__ uint32_t cand_slot(uint32_t k) {
  return (k * 0x9E3779B1u) >> (32 - __builtin_ctz(uint32_t(SLOTS)));
}
template <int SLOTS>
__device__ __forceinline__ uint32_t cand_slot(uint64_t k) {
  return ((uint32_t(k) ^ (uint32_t(k >> 32) * 0x85EBCA77u)) * 0x9E3779B1u) >> (32 - __builtin_ctz(uint32_t(SLOTS)));
}
// The valid candidates into the table, one a thread (their keys are distinct,
// so a slot once taken stays with its key).  One thread inserting all 64
// waited for 128 loads in turn, in every workgroup.
template <int SLOTS, typename K>
__device__ __forceinline__ void cand_insert(const uint64_t* cand_keys, const uint32_t* cand_sample_counts, uint64_t* s_key,
                                            int32_t* s_idx) {
  if (threadIdx.x >= uint32_t(kPlanCand) || cand_sample_counts[threadIdx.x] == 0) return;
  const K key = K(cand_keys[threadIdx.x]);
  uint32_t s = cand_slot<SLOTS>(key);
  while (atomicCAS(&s_idx[s], -1, int32_t(threadIdx.x)) >= 0) s = (s + 1) & uint32_t(SLOTS - 1);
  s_key[s] = uint64_t(key);
}

template <int KB>
__global__ __launch_bounds__(256) void k_count_cand(const void* keys, int64_t n, const uint64_t* cand_keys,
                                                    const uint32_t* cand_sample_counts,
                                                    unsigned long long* counts) {
  using key_t = typename KeyT<KB>::key_t;
  constexpr int SLOTS = 2 * kPlanCand;
  __shared__ uint64_t s_key[SLOTS];
  __shared__ int32_t s_idx[SLOTS];
  __shared__ uint32_t s_cnt[kPlanCand];
  const int tid = threadIdx.x;
  for (int i = tid; i < SLOTS; i += 256) s_idx[i] = -1;
  for (int i = tid; i < kPlanCand; i += 256) s_cnt[i] = 0;
  __syncthreads();
  cand_insert<SLOTS, key_t>(cand_keys, cand_sample_counts, s_key, s_idx);
  __syncthreads();
  const key_t* k = static_cast<const key_t*>(keys);
  for (int64_t i = blockIdx.x * int64_t(256) + tid; i < n; i += int64_t(gridDim.x) * 256) {
    const key_t key = k[i];
    uint64_t v = uint64_t(key);
    if (KB == 4) v &= 0xffffffffull;
    uint32_t s = cand_slot<SLOTS>(key);
    while (s_idx[s] >= 0) {  // at most 64 of the 128 slots are used
      if (s_key[s] == v) {
        atomicAdd(&s_cnt[s_idx[s]], 1u);
        break;
      }
      s = (s + 1) & uint32_t(SLOTS - 1);
    }
  }
  __syncthreads();
  for (int c = tid; c < kPlanCand; c += 256)
    if (s_cnt[c]) atomicAdd(&counts[c], (unsigned long long)s_cnt[c]);
}

// The same count over a 16-byte-aligned column (256M Zipf(1.0) int32 keys: 282
// us with index and key apart and a walk to a free slot, 191 us = 5.6 TB/s
// here), read as 16-byte vectors with
// four loads in flight per thread; the n % (16 / key bytes) last keys are read
// one by one by the first workgroup.  The table has 16 slots per candidate and
// nearly every key is decided by the first one it reads.  Few, large workgroups: each ends with up to 64
// atomic adds to the same counters, which take turns.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kCandBlock = 1024;

template <int KB>
__global__ __launch_bounds__(kCandBlock) void k_count_cand_vec(const void* keys, int64_t n, const uint64_t* cand_keys,
                                                               const uint32_t* cand_sample_counts,
                                                               unsigned long long* counts) {
  using key_t = typename KeyT<KB>::key_t;
  constexpr uint32_t SLOTS = 16 * kPlanCand;
  constexpr int PER = 16 / KB;  // keys per vector
  // a slot's key beside its candidate: index + 1 (0: free), kMore if the next slot is taken
  struct alignas(2 * sizeof(key_t)) Entry {
    key_t key;
    uint32_t cand;
  };
  constexpr uint32_t kMore = 0x80000000u;
  __shared__ Entry s_tab[SLOTS];
  __shared__ uint32_t s_cnt[kPlanCand];
  const int tid = threadIdx.x;
  for (uint32_t i = tid; i < SLOTS; i += kCandBlock) s_tab[i].cand = 0;
  for (int i = tid; i < kPlanCand; i += kCandBlock) s_cnt[i] = 0;
  __syncthreads();
  if (tid < kPlanCand && cand_sample_counts[tid] != 0) {
    const key_t key = key_t(cand_keys[tid]);
    uint32_t s = cand_slot<SLOTS>(key);
    while (atomicCAS(&s_tab[s].cand, 0u, uint32_t(tid) + 1u) != 0u) s = (s + 1u) % SLOTS;
    s_tab[s].key = key;
  }
  __syncthreads();
  uint32_t more = 0;  // SLOTS == kCandBlock: one slot a thread
  static_assert(SLOTS == uint32_t(kCandBlock), "one slot a thread");
  if (s_tab[tid].cand != 0u && s_tab[(uint32_t(tid) + 1u) % SLOTS].cand != 0u) more = kMore;
  __syncthreads();
  s_tab[tid].cand |= more;
  __syncthreads();
  // One read decides nearly every key: a free slot or another key with
  // nothing behind it is no candidate, the same key is counted.  Only a key
  // that meets another one with more behind it walks on.
  auto lookup = [&](key_t key) {
    uint32_t s = cand_slot<SLOTS>(key);
    Entry e = s_tab[s];
    bool hit = e.cand != 0u && e.key == key;
    bool walk = !hit && (e.cand & kMore) != 0u;
    while (walk) {
      s = (s + 1u) % SLOTS;
      e = s_tab[s];
      hit = e.cand != 0u && e.key == key;
      walk = !hit && (e.cand & kMore) != 0u;
    }
    if (hit) atomicAdd(&s_cnt[(e.cand & ~kMore) - 1u], 1u);
  };
  auto lookup_vec = [&](const u32x4 q) {
    if constexpr (KB == 4) {
      lookup(q.x);
      lookup(q.y);
      lookup(q.z);
      lookup(q.w);
    } else {
      lookup(uint64_t(q.x) | (uint64_t(q.y) << 32));
      lookup(uint64_t(q.z) | (uint64_t(q.w) << 32));
    }
  };
  const u32x4* k4 = static_cast<const u32x4*>(keys);
  const int64_t nv = n / PER, stride = int64_t(gridDim.x) * kCandBlock;
  int64_t i = blockIdx.x * int64_t(kCandBlock) + tid;
  for (; i + 3 * stride < nv; i += 4 * stride) {
    const u32x4 a = __builtin_nontemporal_load(k4 + i), b = __builtin_nontemporal_load(k4 + i + stride);
    const u32x4 c = __builtin_nontemporal_load(k4 + i + 2 * stride), d = __builtin_nontemporal_load(k4 + i + 3 * stride);
    lookup_vec(a);
    lookup_vec(b);
    lookup_vec(c);
    lookup_vec(d);
  }
  for (; i < nv; i += stride) lookup_vec(k4[i]);
  if (blockIdx.x == 0 && int64_t(tid) < n - nv * PER) lookup(static_cast<const key_t*>(keys)[nv * PER + tid]);
  __syncthreads();
  for (int c = tid; c < kPlanCand; c += kCandBlock)
    if (s_cnt[c]) atomicAdd(&counts[c], (unsigned long long)s_cnt[c]);
}

hipError_t planner_sketch(const void* keys, int64_t n, int key_bytes, int64_t n_build, float* feat,
                          uint64_t* cand_keys, uint32_t* cand_counts, hipStream_t s) {
  if (key_bytes == 4)
    hipLaunchKernelGGL(k_sketch<4>, dim3(1), dim3(1024), 0, s, keys, n, n_build, feat, cand_keys, cand_counts);
  else
    hipLaunchKernelGGL(k_sketch<8>, dim3(1), dim3(1024), 0, s, keys, n, n_build, feat, cand_keys, cand_counts);
  return hipGetLastError();
}

hipError_t planner_count_candidates(const void* keys, int64_t n, int key_bytes, const uint64_t* cand_keys,
                                    const uint32_t* cand_sample_counts, unsigned long long* counts,
                                    hipStream_t s) {
  hipError_t e = launch_fill_u64(reinterpret_cast<uint64_t*>(counts), 0, kPlanCand, s);
  if (e != hipSuccess || n == 0) return e;
  if (reinterpret_cast<uintptr_t>(keys) % 16 == 0) {
    int64_t g = (n / (16 / key_bytes) + kCandBlock - 1) / kCandBlock;
    if (g < 1) g = 1;
    if (g > 512) g = 512;  // two per CU
    if (key_bytes == 4)
      hipLaunchKernelGGL(k_count_cand_vec<4>, dim3(int(g)), dim3(kCandBlock), 0, s, keys, n, cand_keys, cand_sample_counts,
                         counts);
    else
      hipLaunchKernelGGL(k_count_cand_vec<8>, dim3(int(g)), dim3(kCandBlock), 0, s, keys, n, cand_keys, cand_sample_counts,
                         counts);
    return hipGetLastError();
  }
  int64_t g = (n + 255) / 256;
  if (g > 4096) g = 4096;
  if (key_bytes == 4)
    hipLaunchKernelGGL(k_count_cand<4>, dim3(int(g)), dim3(256), 0, s, keys, n, cand_keys, cand_sample_counts,
                       counts);
  else
    hipLaunchKernelGGL(k_count_cand<8>, dim3(int(g)), dim3(256), 0, s, keys, n, cand_keys, cand_sample_counts,
                       counts);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// MLP kernels
// ---------------------------------------------------------------------------
// C[M x N] = act((accum ? C : 0) + op(A) op(B) + bias), where op(A)(m, k) =
// A[m * sam + k * sak] and op(B)(k, n) = B[k * sbk + n * sbn].  64 x 64 tiles,
// 256 threads with 4 x 4 outputs each, K staged through LDS 16 at a time.
__global__ __launch_bounds__(256) void k_gemm(const float* __restrict__ A, int64_t sam, int64_t sak,
                                              const float* __restrict__ B, int64_t sbk, int64_t sbn, float* C, int M,
                                              int N, int K, const float* bias, int relu, int accum) {
  constexpr int TM = 64, TN = 64, TK = 16;
  __shared__ float As[TK][TM + 4];
  __shared__ float Bs[TK][TN + 4];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
  for (int k0 = 0; k0 < K; k0 += TK) {
    for (int e = threadIdx.x; e < TM * TK; e += 256) {
      const int mm = e / TK, kk = e % TK, m = m0 + mm, k = k0 + kk;
      As[kk][mm] = (m < M && k < K) ? A[int64_t(m) * sam + int64_t(k) * sak] : 0.f;
    }
    for (int e = threadIdx.x; e < TK * TN; e += 256) {
      const int kk = e / TN, nn = e % TN, k = k0 + kk, n = n0 + nn;
      Bs[kk][nn] = (k < K && n < N) ? B[int64_t(k) * sbk + int64_t(n) * sbn] : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
      if (m < M && n < N) {
        float v = acc[i][j];
        if (accum) v += C[int64_t(m) * N + n];
        if (bias) v += bias[n];
        if (relu) v = v > 0.f ? v : 0.f;
        C[int64_t(m) * N + n] = v;
      }
    }
}

static hipError_t gemm(const float* A, int64_t sam, int64_t sak, const float* B, int64_t sbk, int64_t sbn, float* C,
                       int M, int N, int K, const float* bias, bool relu, hipStream_t s) {
  dim3 grid((N + 63) / 64, (M + 63) / 64);
  hipLaunchKernelGGL(k_gemm, grid, dim3(256), 0, s, A, sam, sak, B, sbk, sbn, C, M, N, K, bias, relu ? 1 : 0, 0);
  return hipGetLastError();
}

// db[n] = sum over rows of dY[r][n].
__global__ void k_colsum(const float* dY, int rows, int N, float* db) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= N) return;
  float acc = 0.f;
  for (int r = 0; r < rows; ++r) acc += dY[int64_t(r) * N + n];
  db[n] = acc;
}

// dH[i] = 0 where the ReLU output H[i] is 0.
__global__ void k_relu_mask(float* dH, const float* H, int64_t n) {
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
    if (!(H[i] > 0.f)) dH[i] = 0.f;
}

// Softmax cross-entropy on the bits-1, bits-2 and pass heads and binary
// cross-entropy on the 64 heavy flags; labels[b] = {bits1 class, bits2 class
// or -1 (one pass), pass class}, heavy[b][j] = 1, 0 or -1 (no candidate).
// Writes dOut (mean over the batch) and the mean loss.  One workgroup.
__global__ __launch_bounds__(256) void k_heads_loss(const float* out, const int32_t* labels, const float* heavy,
                                                    int batch, float* dout, float* loss) {
  __shared__ float s_red[256 / kWave];
  float lsum = 0.f;
  const float inv = 1.f / float(batch);
  for (int b = threadIdx.x; b < batch; b += 256) {
    const float* o = out + int64_t(b) * kPlanOut;
    float* g = dout + int64_t(b) * kPlanOut;
    auto ce = [&](int off, int ncls, int label) {
      if (label < 0) {
        for (int c = 0; c < ncls; ++c) g[off + c] = 0.f;
        return 0.f;
      }
      float mx = o[off];
      for (int c = 1; c < ncls; ++c) mx = fmaxf(mx, o[off + c]);
      float z = 0.f;
      for (int c = 0; c < ncls; ++c) z += expf(o[off + c] - mx);
      for (int c = 0; c < ncls; ++c) g[off + c] = (expf(o[off + c] - mx) / z - (c == label ? 1.f : 0.f)) * inv;
      return logf(z) + mx - o[off + label];  // o and g are different buffers
    };
    const int32_t* lb = labels + int64_t(b) * 3;
    float l = ce(0, kPlanBitsCls, lb[0]);
    l += ce(kPlanBitsCls, kPlanBitsCls, lb[1]);
    l += ce(2 * kPlanBitsCls, kPlanPassCls, lb[2]);
    const int hoff = 2 * kPlanBitsCls + kPlanPassCls;
    for (int j = 0; j < kPlanCand; ++j) {
      const float t = heavy[int64_t(b) * kPlanCand + j];
      const float x = o[hoff + j];
      if (t < 0.f) {
        g[hoff + j] = 0.f;
        continue;
      }
      const float p = 1.f / (1.f + expf(-x));
      g[hoff + j] = (p - t) * inv / float(kPlanCand);
      // log(1 + e^-|x|) + max(x, 0) - t x, written to stay finite
      l += (fmaxf(x, 0.f) - t * x + log1pf(expf(-fabsf(x)))) / float(kPlanCand);
    }
    lsum += l;
  }
  for (int d = kWave / 2; d > 0; d >>= 1) lsum += __shfl_xor(lsum, d, kWave);
  if ((threadIdx.x & (kWave - 1)) == 0) s_red[threadIdx.x / kWave] = lsum;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.f;
    for (int w = 0; w < 256 / kWave; ++w) t += s_red[w];
    *loss = t * inv;
  }
}

__global__ void k_adam(float* w, const float* g, float* m, float* v, int64_t n, float lr, float bc1, float bc2) {
  constexpr float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
  }
}

// Scratch (floats): H1, H2, dH2, dH1 [batch x H]; logits and dOut
// [batch x O]; gradients [params].
size_t planner_scratch_floats(int batch) {
  return 4 * size_t(batch) * kPlanHidden + 2 * size_t(batch) * kPlanOut + kPlanParams + 64;
}

static hipError_t forward(const float* w, const float* x, int batch, float* h1, float* h2, float* out,
                          hipStream_t s) {
  const int F = kPlanFeat, H = kPlanHidden, O = kPlanOut;
  hipError_t e = gemm(x, F, 1, w + kPlanW1, H, 1, h1, batch, H, F, w + kPlanB1, true, s);
  if (e == hipSuccess) e = gemm(h1, H, 1, w + kPlanW2, H, 1, h2, batch, H, H, w + kPlanB2, true, s);
  if (e == hipSuccess) e = gemm(h2, H, 1, w + kPlanW3, O, 1, out, batch, O, H, w + kPlanB3, false, s);
  return e;
}

// One sample (planning a join): matrix-vector products split over K, so
// every layer reads its weights with many workgroups.  Workgroup w of a layer
// takes input rows [w * KC, (w + 1) * KC) and writes partial sums part[w][n];
// the next layer first adds its input's partials, the bias and the ReLU.
// Fixed split and summation order: the logits are deterministic.
constexpr int kGemvBlock = 256;
constexpr int kGemvSplit1 = 16, kGemvSplit2 = 8, kGemvSplit3 = 8;

__global__ __launch_bounds__(kGemvBlock) void k_gemv(const float* x, const float* x_parts, int x_nparts,
                                                     const float* x_bias, const float* W, int K, int N, int KC,
                                                     float* out_parts) {
  __shared__ float s_x[128];
  const int k0 = blockIdx.x * KC, k1 = min(K, k0 + KC);
  for (int k = k0 + threadIdx.x; k < k1; k += kGemvBlock) {
    float v;
    if (x_parts) {  // hidden layer input: sum of partials + bias, ReLU
      v = x_bias[k];
      for (int p = 0; p < x_nparts; ++p) v += x_parts[size_t(p) * K + k];
      v = v > 0.f ? v : 0.f;
    } else {
      v = x[k];
    }
    s_x[k - k0] = v;
  }
  __syncthreads();
  for (int n = threadIdx.x; n < N; n += kGemvBlock) {
    float acc = 0.f;
#pragma unroll 16
    for (int k = k0; k < k1; ++k) acc = fmaf(s_x[k - k0], W[size_t(k) * N + n], acc);  // 16 rows' loads together, summed in order (17.8 -> 4.3 us a layer)
    out_parts[size_t(blockIdx.x) * N + n] = acc;
  }
}

__global__ __launch_bounds__(kGemvBlock) void k_gemv_final(const float* parts, int nparts, const float* bias, int N,
                                                           float* out) {
  for (int n = threadIdx.x; n < N; n += kGemvBlock) {
    float v = bias[n];
    for (int p = 0; p < nparts; ++p) v += parts[size_t(p) * N + n];
    out[n] = v;
  }
}

static hipError_t forward_one(const float* w, const float* x, float* out, float* scratch, hipStream_t s) {
  const int F = kPlanFeat, H = kPlanHidden, O = kPlanOut;
  float* p1 = scratch;                                  // [kGemvSplit1][H]
  float* p2 = p1 + size_t(kGemvSplit1) * H;             // [kGemvSplit2][H]
  float* p3 = p2 + size_t(kGemvSplit2) * H;             // [kGemvSplit3][O]
  const int kc1 = (F + kGemvSplit1 - 1) / kGemvSplit1, kc2 = H / kGemvSplit2, kc3 = H / kGemvSplit3;
  hipLaunchKernelGGL(k_gemv, dim3(kGemvSplit1), dim3(kGemvBlock), 0, s, x, nullptr, 0, nullptr, w + kPlanW1, F, H,
                     kc1, p1);
  hipLaunchKernelGGL(k_gemv, dim3(kGemvSplit2), dim3(kGemvBlock), 0, s, nullptr, p1, kGemvSplit1, w + kPlanB1,
                     w + kPlanW2, H, H, kc2, p2);
  hipLaunchKernelGGL(k_gemv, dim3(kGemvSplit3), dim3(kGemvBlock), 0, s, nullptr, p2, kGemvSplit2, w + kPlanB2,
                     w + kPlanW3, H, O, kc3, p3);
  hipLaunchKernelGGL(k_gemv_final, dim3(1), dim3(kGemvBlock), 0, s, p3, kGemvSplit3, w + kPlanB3, O, out);
  return hipGetLastError();
}
static_assert((kPlanFeat + kGemvSplit1 - 1) / kGemvSplit1 <= 128 && kPlanHidden / kGemvSplit2 <= 128,
              "a workgroup's input rows fit its LDS slice");

hipError_t planner_forward(const float* w, const float* x, int batch, float* out, float* scratch, hipStream_t s) {
  if (batch == 1) return forward_one(w, x, out, scratch, s);
  float* h1 = scratch;
  float* h2 = h1 + size_t(batch) * kPlanHidden;
  return forward(w, x, batch, h1, h2, out, s);
}

hipError_t planner_train_step(float* w, float* m, float* v, int step, float lr, const float* x, const int32_t* labels,
                              const float* heavy, int batch, float* loss, float* scratch, hipStream_t s) {
  const int F = kPlanFeat, H = kPlanHidden, O = kPlanOut;
  float* h1 = scratch;
  float* h2 = h1 + size_t(batch) * H;
  float* dh2 = h2 + size_t(batch) * H;
  float* dh1 = dh2 + size_t(batch) * H;
  float* out = dh1 + size_t(batch) * H;
  float* g_out = out + size_t(batch) * O;
  float* grad = g_out + size_t(batch) * O;
  hipError_t e = forward(w, x, batch, h1, h2, out, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_heads_loss, dim3(1), dim3(256), 0, s, out, labels, heavy, batch, g_out, loss);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  // layer 3: dW3 = H2^T dOut, db3 = colsum(dOut), dH2 = dOut W3^T (masked by H2 > 0)
  if ((e = gemm(h2, 1, H, g_out, O, 1, grad + kPlanW3, H, O, batch, nullptr, false, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_colsum, dim3((O + 255) / 256), dim3(256), 0, s, g_out, batch, O, grad + kPlanB3);
  if ((e = gemm(g_out, O, 1, w + kPlanW3, 1, O, dh2, batch, H, O, nullptr, false, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_relu_mask, dim3(64), dim3(256), 0, s, dh2, h2, int64_t(batch) * H);
  // layer 2
  if ((e = gemm(h1, 1, H, dh2, H, 1, grad + kPlanW2, H, H, batch, nullptr, false, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_colsum, dim3((H + 255) / 256), dim3(256), 0, s, dh2, batch, H, grad + kPlanB2);
  if ((e = gemm(dh2, H, 1, w + kPlanW2, 1, H, dh1, batch, H, H, nullptr, false, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_relu_mask, dim3(64), dim3(256), 0, s, dh1, h1, int64_t(batch) * H);
  // layer 1
  if ((e = gemm(x, 1, F, dh1, H, 1, grad + kPlanW1, F, H, batch, nullptr, false, s)) != hipSuccess) return e;
  hipLaunchKernelGGL(k_colsum, dim3((H + 255) / 256), dim3(256), 0, s, dh1, batch, H, grad + kPlanB1);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const double bc1 = 1.0 - std::pow(0.9, double(step)), bc2 = 1.0 - std::pow(0.999, double(step));
  hipLaunchKernelGGL(k_adam, dim3(512), dim3(256), 0, s, w, grad, m, v, int64_t(kPlanParams), lr, float(bc1),
                     float(bc2));
  return hipGetLastError();
}

}  // namespace pj
