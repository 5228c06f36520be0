// pj_wide.h -- the plain join's own pipeline for gfx950 (kernels and launches,
// compiled as part of pj_join.hip): one wide radix pass
// and a join over large LDS tables, or no pass at all for small build tables.
//
//   k_wide_hist     digit counts of both tables, per XCD share of the rows.
//   k_wide_scan     partition starts, the write cursor of every (XCD, digit)
//                   and the join's work items.
//   k_wide_scatter  one pass over up to 4096 digits.  The workgroups of an
//                   XCD share one write cursor per digit, claimed per tile
//                   with one atomic add, so the XCD's tiles complete each
//                   other's 128-byte lines in its L2 while they are there.
//   k_wide_join     per item (partition chunk of up to 17408 build tuples,
//                   probe slice): the chunk is sorted into hash buckets in
//                   LDS, probes read their bucket's entries, and each round
//                   claims exactly the output it writes.
//
// Digit and bucket come from one multiplicative hash of the key: the digit is
// its top bits, the bucket the bits below them, so neither strided nor dense
// keys crowd a partition or a bucket.
#pragma once
#include <cmath>

#include "pj_device.h"
#include "pj_internal.h"

namespace pj {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Partitioned tuples: 8 bytes, or 12 with 8-byte keys (three words, loaded and
// stored as one access each: the scatter of 16M x 64M rows takes 366 us and
// the join 487; with a fourth, empty word they took 437 and 516).
struct __attribute__((packed, aligned(4))) Tup12 {
  uint32_t x, y, z;
};
template <int KB> struct WideTup;
template <> struct WideTup<4> {
  using type = uint2;
  __device__ __forceinline__ static type make(uint32_t k, int32_t p) { return make_uint2(k, uint32_t(p)); }
  __device__ __forceinline__ static uint32_t key(const type& t) { return t.x; }
  __device__ __forceinline__ static int32_t pay(const type& t) { return int32_t(t.y); }
};
template <> struct WideTup<8> {
  using type = Tup12;
  __device__ __forceinline__ static type make(uint64_t k, int32_t p) {
    return type{uint32_t(k), uint32_t(k >> 32), uint32_t(p)};
  }
  __device__ __forceinline__ static uint64_t key(const type& t) { return uint64_t(t.x) | (uint64_t(t.y) << 32); }
  __device__ __forceinline__ static int32_t pay(const type& t) { return int32_t(t.z); }
};
constexpr size_t wide_tuple_bytes(int key_bytes) { return key_bytes == 4 ? 8 : 12; }

// A bijection of 4-byte keys.  Dense keys spread more evenly over the buckets
// than random ones under the multiplication; the shift leaves them so and
// breaks up the strides (3, 4, 8, 12, ...) whose multiples fall together in a
// few buckets otherwise (4M keys of stride 4: 0.73 of them in buckets of more
// than four, now none; random keys 0.02).
__device__ __forceinline__ uint32_t wide_hash(uint32_t k) { return (k ^ (k >> 15)) * 0x9E3779B1u; }
__device__ __forceinline__ uint32_t wide_hash(uint64_t k) {
  return wide_hash(uint32_t(k) ^ (uint32_t(k >> 32) * 0x85EBCA77u));
}
// Top `bits` bits of a hash (0 bits: 0).
__device__ __forceinline__ uint32_t top_bits(uint32_t h, int bits) { return bits ? h >> (32 - bits) : 0u; }

// Inclusive prefix sum over the 64 lanes of a wave with DPP moves.
__device__ __forceinline__ uint32_t wave_scan(uint32_t x) {
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x111, 0xf, 0xf, false));  // row_shr:1
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x112, 0xf, 0xf, false));  // row_shr:2
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x114, 0xf, 0xf, false));  // row_shr:4
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x118, 0xf, 0xf, false));  // row_shr:8
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x142, 0xa, 0xf, false));  // row_bcast:15
  x += uint32_t(__builtin_amdgcn_update_dpp(0, int(x), 0x143, 0xc, 0xf, false));  // row_bcast:31
  return x;
}

__device__ __forceinline__ uint32_t sgpr(uint32_t x) { return uint32_t(__builtin_amdgcn_readfirstlane(int(x))); }

// Empty asm that takes a register as read and rewritten: a load into it is
// waited for here.
__device__ __forceinline__ void pin(uint32_t& v) { __asm__ volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin(uint64_t& v) { __asm__ volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin(int32_t& v) { __asm__ volatile("" : "+v"(v)); }

// The thread index through an opaque move, once per phase: row numbers formed
// from it are then computed where they are used instead of being kept in
// registers, which run out.
__device__ __forceinline__ uint32_t opaque_tid() {
  uint32_t t;
  __asm__ volatile("v_mov_b32 %0, %1" : "=v"(t) : "v"(uint32_t(threadIdx.x)));
  return t;
}

constexpr int kWideBlock = 1024;  // histogram and scatter workgroup

// ---------------------------------------------------------------------------
// k_wide_hist: rows are dealt to the XCD shares in tiles of `tile` rows (tile
// t to share t % 8), as the scatter takes them.  Workgroups [0, g0) serve
// table 0, the others table 1.  cnt[table][share][digit] is zero on entry.
// Bound by reading the keys once: 64M x 256M int32 211 us, 1.34 GB at 6.4 TB/s
// (257 us before, with one workgroup to a CU and a [segment][digit] matrix to
// write); two workgroups a CU need its bins at 16 KB each.
// ---------------------------------------------------------------------------
template <int KB, bool VEC>
__global__ __launch_bounds__(kWideBlock) void k_wide_hist(WideArgs A, uint32_t g0) {
  extern __shared__ uint32_t s_bins[];
  const int tid = threadIdx.x;
  const uint32_t tb = blockIdx.x >= g0 ? 1u : 0u;
  const uint32_t local = tb ? blockIdx.x - g0 : blockIdx.x, groups = tb ? gridDim.x - g0 : g0;
  const uint32_t x = local % kNumXcd, n = A.n[tb], tile = A.tile, nt = (n + tile - 1) / tile;
  const int P = 1 << A.bits, bits = A.bits;
  if (local >= nt) return;
  using key_t = typename KeyT<KB>::key_t;
  const key_t* keys = static_cast<const key_t*>(A.keys[tb]);
  for (int i = tid; i < P; i += kWideBlock) s_bins[i] = 0;
  lds_barrier();
  // Under a heavy key same-address LDS adds serialise: when kHeavyLanes or
  // more lanes of a wave's first key share lane 0's digit, each row counts
  // its lanes with that digit with one add.
  auto count4 = [&](const uint32_t (&d)[4]) {
    const uint32_t f = sgpr(d[0]);
    if (__popcll(__ballot(d[0] == f)) >= kHeavyLanes) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint64_t same = __ballot(d[c] == f);
        const uint32_t inc = d[c] != f ? 1u : (mbcnt(same) == 0u ? uint32_t(__popcll(same)) : 0u);
        if (inc) atomicAdd(&s_bins[d[c]], inc);
      }
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) atomicAdd(&s_bins[d[c]], 1u);
    }
  };
  for (uint32_t t = local; t < nt; t += groups) {  // groups is a multiple of 8: the share stays x
    const uint32_t lo = t * tile, hi = min(n, lo + tile);
    uint32_t i = lo;
    if (VEC) {
      constexpr uint32_t STEP = 4 * kWideBlock;
      for (; i + 4 * STEP <= hi; i += 4 * STEP) {  // 16 keys a thread: the loads are issued together
        uint32_t d[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const key_t* p = keys + i + u * STEP + tid * 4;
          if constexpr (KB == 4) {
            const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
            d[u][0] = top_bits(wide_hash(v.x), bits); d[u][1] = top_bits(wide_hash(v.y), bits);
            d[u][2] = top_bits(wide_hash(v.z), bits); d[u][3] = top_bits(wide_hash(v.w), bits);
          } else {
            const u32x4 a = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
            const u32x4 b = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + 2));
            d[u][0] = top_bits(wide_hash(uint64_t(a.x) | (uint64_t(a.y) << 32)), bits);
            d[u][1] = top_bits(wide_hash(uint64_t(a.z) | (uint64_t(a.w) << 32)), bits);
            d[u][2] = top_bits(wide_hash(uint64_t(b.x) | (uint64_t(b.y) << 32)), bits);
            d[u][3] = top_bits(wide_hash(uint64_t(b.z) | (uint64_t(b.w) << 32)), bits);
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) count4(d[u]);
      }
    }
    for (; i + 4 * kWideBlock <= hi; i += 4 * kWideBlock) {
      uint32_t d[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) d[c] = top_bits(wide_hash(__builtin_nontemporal_load(keys + i + c * kWideBlock + tid)), bits);
      count4(d);
    }
    for (; i < hi; i += kWideBlock)
      if (i + tid < hi) atomicAdd(&s_bins[top_bits(wide_hash(keys[i + tid]), bits)], 1u);
  }
  lds_barrier();
  uint32_t* row = A.cnt + size_t(tb * kNumXcd + x) * P;
  for (int i = tid; i < P; i += kWideBlock) {
    const uint32_t v = s_bins[i];
    if (v) atomicAdd(&row[i], v);
  }
}

// ---------------------------------------------------------------------------
// k_wide_scan: one thread per digit.  Each block of kWideScan digits scans
// its own totals and leaves the block sums for the consumers to add (at most
// 16 blocks): start[table][digit] and cnt[table][share][digit], which becomes
// the share's write cursor, are relative to the block.  The join's items of a
// partition are its build chunks times its probe slices.  Also clears the pair
// count.  A latency chain of a few loads: 5 us at 4096 digits (the column and
// offset scans it stands for took 37 us at 64M x 256M).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kWideScan) void k_wide_scan(WideArgs A) {
  __shared__ uint32_t s_tmp[3][kWideScan / kWave + 1];
  const uint32_t P = 1u << A.bits, d = blockIdx.x * kWideScan + threadIdx.x;
  uint32_t tot[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    uint32_t c[kNumXcd], sum = 0, total;
    uint32_t* cnt = A.cnt + size_t(t) * kNumXcd * P + d;
#pragma unroll
    for (int x = 0; x < kNumXcd; ++x) {
      c[x] = d < P ? cnt[size_t(x) * P] : 0u;
      sum += c[x];
    }
    tot[t] = sum;
    uint32_t run = block_exclusive_scan<kWideScan>(d < P ? sum + A.pad[t] : 0u, s_tmp[t], &total);
    if (d < P) {
      A.start[t][d] = run;
#pragma unroll
      for (int x = 0; x < kNumXcd; ++x) {
        cnt[size_t(x) * P] = run;
        run += c[x];
      }
    }
    if (threadIdx.x == 0) A.bsum[t * kWideScanMax + blockIdx.x] = total;
  }
  const uint32_t items = tot[0] && tot[1] ? ((tot[0] - 1) / A.cap + 1) * ((tot[1] - 1) / A.slice + 1) : 0u;
  uint32_t total;
  const uint32_t run = block_exclusive_scan<kWideScan>(items, s_tmp[2], &total);
  A.iscan[d] = run;  // kWideScan entries per block, whatever P
  if (threadIdx.x == 0) {
    A.bsum[2 * kWideScanMax + blockIdx.x] = total;
    if (blockIdx.x == 0) {
      A.bsum[3 * kWideScanMax] = 0;  // the join's item tickets
      *A.d_count = 0ull;
    }
  }
}

// Exclusive prefix sums of the three rows of block sums into s_pre[row][0 ..
// nblk] by the first wave.  The caller synchronises.
__device__ __forceinline__ void block_prefixes(const WideArgs& A, uint32_t (*s_pre)[kWideScanMax + 1]) {
  if (threadIdx.x < kWave) {
    const uint32_t lane = threadIdx.x, nblk = ((1u << A.bits) + kWideScan - 1) / kWideScan;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const uint32_t inc = wave_scan(lane < nblk ? A.bsum[r * kWideScanMax + lane] : 0u);
      if (lane == 0) s_pre[r][0] = 0;
      if (lane < uint32_t(kWideScanMax)) s_pre[r][lane + 1] = inc;
    }
  }
}

// ---------------------------------------------------------------------------
// k_wide_scatter: tiles of E * 1024 rows of both tables (table 0's first), in
// the histogram's shares.  A tile is counted by digit in LDS (two 16-bit
// counts a word), each digit's rows take their place in the share's run of
// that digit with one global atomic add, the tile is staged in digit order
// and stored.  The runs of one tile are a few tuples long, but the tiles of
// an XCD fill the same lines one after another within its L2, which writes
// them back whole.
// Bound by memory, and by what its writes add to it: 64M x 256M 1.19 ms for
// 1.34 GB read and 2.68 GB of tuples, of which 3.45 GB reach memory (each
// atomic writes its line of cursors through, and some lines leave the L2
// unfinished at 4096 digits); the two passes it stands for took 2.19 ms.  The
// cost of a digit count on random keys, 256M tuples: 512 digits 0.69 ms, 2048
// 0.74, 4096 0.92.  16K-tuple tiles: runs of 4 tuples at 4096 digits; tiles of
// 8K with two workgroups to a CU were slower, and so were claims after the
// staging (1223 -> 1295 us) and stores kept back until the next tile's staging
// (1441 us).  The cursor adds of two digits at once: 1223 -> 1205 us.
// ---------------------------------------------------------------------------
template <int KB, int E, bool PAY>
__global__ __launch_bounds__(kWideBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_wide_scatter(WideArgs A) {
  using V = typename WideTup<KB>::type;
  using key_t = typename KeyT<KB>::key_t;
  constexpr uint32_t BLOCK = kWideBlock, TILE = BLOCK * E;
  constexpr int NW = kWideBlock / kWave;
  constexpr int WPT = kMaxRadix / 2 / kWideBlock;  // count words per thread, at most
  extern __shared__ __align__(16) uint8_t s_raw[];
  __shared__ uint32_t s_wsum[NW];
  __shared__ uint32_t s_pre[3][kWideScanMax + 1];
  V* s_stage = reinterpret_cast<V*>(s_raw);
  const uint32_t P = 1u << A.bits, W = P / 2;
  const int shift = 32 - A.bits;  // at most 31: there is a digit
  uint32_t* s_cnt = reinterpret_cast<uint32_t*>(s_raw + size_t(TILE) * sizeof(V));  // W words: counts, then stage starts
  uint32_t* s_delta = s_cnt + W;                                                    // P words: output minus stage position
  const uint32_t wave = sgpr(threadIdx.x / kWave);
  const uint32_t x = blockIdx.x % kNumXcd, G = gridDim.x;  // G is a multiple of 8
  const uint32_t nt0 = (A.n[0] + TILE - 1) / TILE, nt0r = (nt0 + kNumXcd - 1) / kNumXcd * kNumXcd;
  const uint32_t nt1 = (A.n[1] + TILE - 1) / TILE;
  const uint32_t nt = nt0r + nt1;  // tiles [nt0, nt0r) are empty, so that a tile's share is its index modulo 8
  block_prefixes(A, s_pre);
  for (uint32_t i = threadIdx.x; i < W; i += BLOCK) s_cnt[i] = 0;

  key_t key[E];
  int32_t pay[E];
  auto load = [&](uint32_t t) {
    const uint32_t tb = t >= nt0r ? 1u : 0u, n = A.n[tb], lo = (t - (tb ? nt0r : 0u)) * TILE;
    const uint32_t tid = opaque_tid(), last = n - lo - 1u;
    const key_t* keys = static_cast<const key_t*>(A.keys[tb]) + lo;  // a scalar row start and 32-bit lane offsets
#pragma unroll
    for (int e = 0; e < E; ++e) key[e] = __builtin_nontemporal_load(keys + min(uint32_t(e) * BLOCK + tid, last));
    if (PAY && A.pay[tb]) {
      const int32_t* p = A.pay[tb] + lo;
#pragma unroll
      for (int e = 0; e < E; ++e) pay[e] = __builtin_nontemporal_load(p + min(uint32_t(e) * BLOCK + tid, last));
    }
  };
  auto next_tile = [&](uint32_t t) {
    t += G;
    return t >= nt0 && t < nt0r ? t + G : t;
  };
  uint32_t t = blockIdx.x;
  if (t >= nt0 && t < nt0r) t += G;
  if (t < nt) load(t);
  lds_barrier();
  while (t < nt) {
    const uint32_t tb = t >= nt0r ? 1u : 0u, n = A.n[tb], lo = (t - (tb ? nt0r : 0u)) * TILE;
    const uint32_t len = min(TILE, n - lo);
    unsigned long long* cursor = reinterpret_cast<unsigned long long*>(A.cnt + size_t(tb * kNumXcd + x) * P);
    // digit << 16 | rank within it
    uint32_t pk[E];
    {
      const uint32_t tid = opaque_tid();
      const uint32_t d0 = wide_hash(key[0]) >> shift;
      // same-address LDS adds serialise: under a heavy key each row's lanes
      // with lane 0's digit rank with one add
      const bool heavy = __popcll(__ballot(d0 == sgpr(d0))) >= kHeavyLanes;
      if (!heavy && len == TILE) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const uint32_t d = wide_hash(key[e]) >> shift, sh = (d & 1u) << 4;
          pk[e] = (d << 16) | ((atomicAdd(&s_cnt[d >> 1], 1u << sh) >> sh) & 0xFFFFu);
        }
      } else {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const uint32_t d = wide_hash(key[e]) >> shift, sh = (d & 1u) << 4;
          const bool valid = e * BLOCK + tid < len;
          const uint32_t f = sgpr(d);
          const uint64_t same = __ballot(valid && d == f);
          const uint32_t k = mbcnt(same);
          uint32_t old = 0;
          const bool mine = valid && d == f;
          if (valid && (!mine || k == 0u)) old = atomicAdd(&s_cnt[d >> 1], (mine ? uint32_t(__popcll(same)) : 1u) << sh);
          old = (old >> sh) & 0xFFFFu;
          // the first of the lanes with digit f holds their first rank
          const uint32_t first = same ? uint32_t(__builtin_ctzll(same)) : 0u;
          const uint32_t fbase = uint32_t(__shfl(int(old), int(first), kWave));
          pk[e] = (d << 16) | (mine ? fbase + k : old);
        }
      }
    }
    lds_barrier();
    // Stage and output ranges of this thread's digits, 2 per count word.  The
    // two digits' cursors advance in one 64-bit add (a cursor stays below
    // 2^32, so nothing carries into the second): every line of cursors an add
    // touches is written through to memory, half the adds write half as much.
    const uint32_t tid = opaque_tid();
    uint32_t c[WPT], mine = 0;
    unsigned long long g[WPT];
#pragma unroll
    for (int k = 0; k < WPT; ++k) {
      c[k] = tid + k * BLOCK < W ? s_cnt[tid + k * BLOCK] : 0u;
      mine += (c[k] & 0xFFFFu) + (c[k] >> 16);
    }
#pragma unroll
    for (int k = 0; k < WPT; ++k) {
      g[k] = 0;
      if (c[k]) g[k] = atomicAdd(cursor + tid + k * BLOCK, (unsigned long long)(c[k] & 0xFFFFu) | ((unsigned long long)(c[k] >> 16) << 32));
    }
    const uint32_t inc = wave_scan(mine);
    if ((tid & (kWave - 1)) == kWave - 1) s_wsum[wave] = inc;
    lds_barrier();
    uint32_t run = inc - mine;
#pragma unroll
    for (int w = 0; w < NW; ++w) run += w < int(wave) ? sgpr(s_wsum[w]) : 0u;
#pragma unroll
    for (int k = 0; k < WPT; ++k)
      if (tid + k * BLOCK < W) {
        const uint32_t a = c[k] & 0xFFFFu, b = c[k] >> 16;
        c[k] = run | ((run + a) << 16);
        s_cnt[tid + k * BLOCK] = c[k];
        run += a + b;
      }
    lds_barrier();
    const uint32_t tid_s = opaque_tid();
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const uint32_t i = e * BLOCK + tid_s;
      if (i < len) {
        const uint32_t d = pk[e] >> 16;
        const int32_t p = PAY && A.pay[tb] ? pay[e] : int32_t(lo + i);
        s_stage[((s_cnt[d >> 1] >> ((d & 1u) << 4)) & 0xFFFFu) + (pk[e] & 0xFFFFu)] = WideTup<KB>::make(key[e], p);
      }
    }
#pragma unroll
    for (int k = 0; k < WPT; ++k)
      if (tid + k * BLOCK < W) {
        const uint32_t d = 2u * (tid + k * BLOCK), pre = s_pre[tb][d / kWideScan];
        s_delta[d] = uint32_t(g[k]) + pre - (c[k] & 0xFFFFu);
        s_delta[d + 1] = uint32_t(g[k] >> 32) + pre - (c[k] >> 16);
      }
    // the next tile's loads are in flight during the flush (the last tile's
    // are read again rather than branch)
    const uint32_t tn = next_tile(t);
    load(tn < nt ? tn : t);
    lds_barrier();
    // Every position is below n with exact counts; the clamp keeps the stores
    // of a full tile unconditional, so that the next wait for the loads does
    // not wait for them.
    V* out = static_cast<V*>(A.tup[tb]);
    const uint32_t end = n + P * A.pad[tb] - 1u;
    const uint32_t tid_f = opaque_tid();
    if (len == TILE) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const uint32_t q = e * BLOCK + tid_f;
        const V v = s_stage[q];
        const uint32_t p = s_delta[wide_hash(WideTup<KB>::key(v)) >> shift] + q;
        out[min(p, end)] = v;
      }
    } else {
      for (uint32_t q = tid_f; q < len; q += BLOCK) {
        const V v = s_stage[q];
        const uint32_t p = s_delta[wide_hash(WideTup<KB>::key(v)) >> shift] + q;
        out[min(p, end)] = v;
      }
    }
    for (uint32_t i = tid_f; i < W; i += BLOCK) s_cnt[i] = 0;
    lds_barrier();
    t = tn;
  }
}

// ---------------------------------------------------------------------------
// k_wide_join
// ---------------------------------------------------------------------------
constexpr uint32_t kWideSpare = 8;

struct WideItem {
  uint32_t rlo, rhi, slo, shi;
};

// The byte at each position of x that is zero: bit 7 of that byte.
__device__ __forceinline__ uint32_t zero_bytes(uint32_t x) {
  const uint32_t t = ((x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | x;
  return ~t & 0x80808080u;
}

// Build: every tuple of the chunk (at most CAP = BLOCK * NB, NB per thread in
// registers) counts into one of 2^LGB buckets and keeps its rank there, the
// counts are scanned, and the tuples are written to LDS in bucket order: a
// dense table without empty slots, so the whole of the LDS holds tuples, and
// without a reserved key.  Each entry has an 8-bit tag, the hash bits that
// follow the digit's and the bucket's.
// Probe: a bucket's entries lie between its start and the next bucket's (one
// entry a bucket on average, at the largest chunks).  One unaligned window of
// four tags is compared with the probe's at once; the few probes whose bucket
// holds more than four entries, or where more than one tag fits, walk their
// bucket.  VERIFY: the tag does not identify the key within its bucket, so the
// table holds the keys too and a tag's match is checked; otherwise
// (4-byte keys and at most 8 hash bits left, the hash being a bijection of the
// key) digit, bucket and tag are the whole key.
// A round probes U tuples per thread; its matches stay in registers while the
// workgroup's pair count is claimed with one global atomic, and are stored
// during the next round, whose probes hide the claim.  A round in which some
// probe matches twice walks its buckets again to write them.
// COLS: no partitions (bits == 0): both sides are read from the key columns.
// Bound by memory under many probes a build row (16M x 256M Zipf: 4.3 GB in
// 1.02 ms, 4.2 TB/s, against 0.94 ms in smaller tables before), otherwise by
// the build of an item, about 17 us for 16384 tuples with nothing else on the
// CU (64M x 256M: 0.94 ms, of which 0.27 the builds; with walks of
// {key, payload} entries in place of the tags 1.68 ms).  Repeated build keys
// are bound by the walks and the uncoalesced stores of their rounds: 12M x 24M
// with keys four times 414 us, of which 230 those two; their pairs read a
// window at a time took registers that spilled (64M x 256M 1.24 ms).
template <int KB, int BLOCK, int NB, int U, int LGB, bool VERIFY, bool COLS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4))) void k_wide_join(WideArgs A) {
  using key_t = typename KeyT<KB>::key_t;
  using V = typename WideTup<KB>::type;
  constexpr uint32_t CAP = uint32_t(BLOCK) * NB, NBK = 1u << LGB, ROUND = uint32_t(BLOCK) * U;
  constexpr int NW = BLOCK / kWave;
  constexpr uint32_t WPT = NBK / 2 / BLOCK;  // bucket words per thread
  static_assert(WPT >= 1 && WPT * BLOCK * 2 == NBK, "whole bucket words per thread");
  static_assert(CAP < 65536 && CAP % 8 == 0 && kWideSpare % 4 == 0, "bucket starts are 16-bit, arrays aligned");
  static_assert(VERIFY || KB == 4, "8-byte keys are compared");
  extern __shared__ __align__(16) uint8_t s_raw[];
  // keys (VERIFY), payloads, bucket starts (two to a word, and the end), tags; kWideSpare entries past the last one
  key_t* s_key = reinterpret_cast<key_t*>(s_raw);
  int32_t* s_pay = reinterpret_cast<int32_t*>(s_raw + (VERIFY ? size_t(CAP + kWideSpare) * KB : 0));
  uint32_t* s_off = reinterpret_cast<uint32_t*>(s_pay + CAP + kWideSpare);  // 16-byte aligned
  uint8_t* s_tag = reinterpret_cast<uint8_t*>(s_off + NBK / 2 + 2);
  __shared__ uint32_t s_wsum[NW];
  __shared__ uint32_t s_wtot[2][NW];
  __shared__ uint64_t s_base[2];
  __shared__ uint32_t s_next;
  __shared__ uint32_t s_pre[3][kWideScanMax + 1];
  const uint32_t wave = sgpr(threadIdx.x / kWave);
  const int bits = COLS ? 0 : A.bits;
  const uint32_t grid = gridDim.x;
  const bool first_only = A.unique != 0;
  const uint64_t capacity = A.capacity;

  if (!COLS) {
    block_prefixes(A, s_pre);
    lds_barrier();
  }
  const uint32_t nblk = COLS ? 1u : ((1u << bits) + kWideScan - 1) / kWideScan;
  const uint32_t total_items = COLS ? (A.n[1] - 1) / A.slice + 1 : sgpr(s_pre[2][nblk]);

  // The partition, chunk and slice of an item: its scan block from the block
  // prefixes, its digit from the block's 256 item starts (4 a lane), then the
  // partition's bounds.
  auto decode = [&](uint32_t item) {
    WideItem w;
    if (COLS) {
      w.rlo = 0;
      w.rhi = A.n[0];
      w.slo = item * A.slice;
      w.shi = min(A.n[1], w.slo + A.slice);
      return w;
    }
    const uint32_t bp_ = lane_id() < nblk ? s_pre[2][lane_id()] : 0xFFFFFFFFu;
    const uint32_t blk = uint32_t(__popcll(__ballot(bp_ <= item))) - 1u;
    const uint32_t local = item - sgpr(s_pre[2][blk]);
    const uint4 v = *reinterpret_cast<const uint4*>(A.iscan + blk * kWideScan + 4 * lane_id());
    const uint32_t below = uint32_t(__popcll(__ballot(v.x <= local)) + __popcll(__ballot(v.y <= local)) +
                                    __popcll(__ballot(v.z <= local)) + __popcll(__ballot(v.w <= local))) - 1u;
    const uint32_t q = blk * kWideScan + below, P = 1u << bits;
    const uint32_t first = sgpr(A.iscan[q]);
    const uint32_t r0 = sgpr(A.start[0][q]) + sgpr(s_pre[0][blk]), s0 = sgpr(A.start[1][q]) + sgpr(s_pre[1][blk]);
    const uint32_t qn = q + 1, bn = qn / kWideScan;
    const uint32_t r1 = (qn < P ? sgpr(A.start[0][qn]) + sgpr(s_pre[0][bn]) : sgpr(s_pre[0][nblk])) - A.pad[0];
    const uint32_t s1 = (qn < P ? sgpr(A.start[1][qn]) + sgpr(s_pre[1][bn]) : sgpr(s_pre[1][nblk])) - A.pad[1];
    const uint32_t ns = (s1 - s0 - 1) / A.slice + 1, k = local - first;
    w.rlo = r0 + (k / ns) * A.cap;
    w.rhi = min(r1, w.rlo + A.cap);
    w.slo = s0 + (k % ns) * A.slice;
    w.shi = min(s1, w.slo + A.slice);
    return w;
  };

  // Row k of a thread is lo + k * BLOCK + tid; rows past the range's end read
  // its last one again (one line for the whole wave) rather than branch: with
  // a branch a row, the compiler moved each row's registers at the branch's
  // end, which waits for its load (the build of 16384 tuples took 30 us).
  // `lo` is a scalar, so that a lane's address is one 32-bit offset.
  auto load_row = [&](int side, uint32_t lo, uint32_t hi, uint32_t tid, key_t& k, int32_t& p) {
    const uint32_t i = min(lo + tid, hi - 1u);
    if constexpr (COLS) {
      k = static_cast<const key_t*>(A.keys[side])[i];
      p = A.pay[side] ? A.pay[side][i] : int32_t(i);
    } else {
      const V v = static_cast<const V*>(A.tup[side])[i];
      k = WideTup<KB>::key(v);
      p = WideTup<KB>::pay(v);
    }
  };
  key_t bk[NB];
  int32_t bp[NB];
  auto load_build = [&](const WideItem& w) {
    const uint32_t tid = opaque_tid();
#pragma unroll
    for (int k = 0; k < NB; ++k) load_row(0, w.rlo + uint32_t(k) * BLOCK, w.rhi, tid, bk[k], bp[k]);
  };
  // Brings the chunk's lines into the L2 while the last item's matches go out:
  // one load of a word per line, whose value nobody reads.  (Loading the
  // tuples themselves there costs twice the registers there are.)
  auto touch_build = [&](const WideItem& w) {
    if constexpr (!COLS) {
      const char* at = static_cast<const char*>(A.tup[0]) + size_t(w.rlo) * sizeof(V);
      const uint32_t bytes = (w.rhi - w.rlo) * uint32_t(sizeof(V));
      for (uint32_t o = opaque_tid() * 128u; o < bytes; o += uint32_t(BLOCK) * 128u)
        (void)*reinterpret_cast<const volatile uint32_t*>(at + o);
    }
  };
  key_t pk[U], nk[U];
  int32_t pp[U], np[U];
  auto load_probe = [&](uint32_t r0, uint32_t shi, key_t (&k_)[U], int32_t (&p_)[U]) {
    const uint32_t tid = opaque_tid();
#pragma unroll
    for (int k = 0; k < U; ++k) load_row(1, r0 + uint32_t(k) * BLOCK, shi, tid, k_[k], p_[k]);
  };
  auto bucket_of = [&](uint32_t h) { return (h << bits) >> (32 - LGB); };
  auto tag_of = [&](uint32_t h) { return (h << (bits + LGB)) >> 24; };
  // Bucket bounds: start in the low half, end in the high half.
  auto bounds_of = [&](uint32_t h) {
    const uint32_t b2 = 2u * bucket_of(h);
    const uint32_t* w = reinterpret_cast<const uint32_t*>(reinterpret_cast<const uint8_t*>(s_off) + (b2 & ~3u));
    return uint32_t(__builtin_amdgcn_alignbyte(w[1], w[0], b2));
  };
  // Whether entry i holds key k with hash h, all of whose bucket's keys share its bucket.
  auto entry_is = [&](uint32_t i, key_t k, uint32_t h) {
    if constexpr (VERIFY) return s_key[i] == k;
    else return uint32_t(s_tag[i]) == tag_of(h);
  };

  uint32_t item = blockIdx.x;
  if (item >= total_items) return;
  WideItem w = decode(item);
  uint32_t par = 0;  // parity of the round: which s_wtot / s_base slot
  while (true) {
    // ---- build
    const uint32_t c = w.rhi - w.rlo;
    uint32_t ticket = 0;  // thread 0: the next item, taken now and read after the item's last round
    {
      const uint32_t tid = opaque_tid();
      if (!COLS && tid == 0) ticket = grid + atomicAdd(A.bsum + 3 * kWideScanMax, 1u);
      load_build(w);
#pragma unroll
      for (uint32_t i = 0; i < WPT; ++i) s_off[tid + i * BLOCK] = 0;
      lds_barrier();
      uint32_t rk[(NB + 1) / 2];
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        if ((k & 1) == 0) rk[k / 2] = 0;
        if (uint32_t(k) * BLOCK + tid < c) {
          const uint32_t b = bucket_of(wide_hash(bk[k])), sh = (b & 1u) << 4;
          const uint32_t r = (atomicAdd(&s_off[b >> 1], 1u << sh) >> sh) & 0xFFFFu;
          rk[k / 2] |= (k & 1) ? r << 16 : r;
        }
      }
      // the first probe round is on its way during the scan and the writes
      // (any earlier its registers are one too many)
      load_probe(w.slo, w.shi, pk, pp);
      lds_barrier();
      {
        // this thread's words, 16 bytes at a time where there are four
        uint32_t v[WPT], sum = 0;
        if constexpr (WPT % 4 == 0) {
#pragma unroll
          for (uint32_t i = 0; i < WPT / 4; ++i) {
            const u32x4 q = reinterpret_cast<const u32x4*>(s_off)[tid * (WPT / 4) + i];
            v[4 * i] = q.x; v[4 * i + 1] = q.y; v[4 * i + 2] = q.z; v[4 * i + 3] = q.w;
          }
        } else {
#pragma unroll
          for (uint32_t i = 0; i < WPT; ++i) v[i] = s_off[tid * WPT + i];
        }
#pragma unroll
        for (uint32_t i = 0; i < WPT; ++i) sum += (v[i] & 0xFFFFu) + (v[i] >> 16);
        const uint32_t inc = wave_scan(sum);
        if ((tid & (kWave - 1)) == kWave - 1) s_wsum[wave] = inc;
        lds_barrier();
        uint32_t run = inc - sum;
#pragma unroll
        for (int i = 0; i < NW; ++i) run += i < int(wave) ? sgpr(s_wsum[i]) : 0u;
#pragma unroll
        for (uint32_t i = 0; i < WPT; ++i) {
          const uint32_t a = v[i] & 0xFFFFu, b = v[i] >> 16;
          v[i] = run | ((run + a) << 16);
          run += a + b;
        }
        if constexpr (WPT % 4 == 0) {
#pragma unroll
          for (uint32_t i = 0; i < WPT / 4; ++i)
            reinterpret_cast<u32x4*>(s_off)[tid * (WPT / 4) + i] = u32x4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
        } else {
#pragma unroll
          for (uint32_t i = 0; i < WPT; ++i) s_off[tid * WPT + i] = v[i];
        }
        if (tid == 0) s_off[NBK / 2] = c;
      }
      lds_barrier();
#pragma unroll
      for (int k = 0; k < NB; ++k)
        if (uint32_t(k) * BLOCK + tid < c) {
          pin(bk[k]);  // the hash is formed again rather than kept across the scan
          const uint32_t h = wide_hash(bk[k]), b = bucket_of(h);
          const uint32_t i = ((s_off[b >> 1] >> ((b & 1u) << 4)) & 0xFFFFu) + ((rk[k / 2] >> ((k & 1) * 16)) & 0xFFFFu);
          if constexpr (VERIFY) s_key[i] = bk[k];
          s_pay[i] = bp[k];
          s_tag[i] = uint8_t(tag_of(h));
        }
      lds_barrier();
    }

    // ---- probe
    bool pending = false;  // a round's matches are held, to be stored
    uint64_t h_m[U];       // its matches: a lane mask per probe row
    uint32_t h_pre = 0, h_n = 0;  // the pairs of the waves before this one, and of this wave
    int32_t h_b[U], h_p[U];
    uint64_t claim = 0;    // thread 0: the claimed position (the atomic's result, read a round later)
    // The wave's matches m[k] as rows of consecutive pairs from position `at` on.
    auto store_rows = [&](uint64_t at, uint32_t n, const uint64_t (&m)[U], const int32_t (&b)[U], const int32_t (&p)[U]) {
      if (at + n <= capacity) {
        uint2* o = reinterpret_cast<uint2*>(A.out) + at;
#pragma unroll
        for (int k = 0; k < U; ++k) {
          if ((m[k] >> lane_id()) & 1u) o[mbcnt(m[k])] = make_uint2(uint32_t(b[k]), uint32_t(p[k]));
          o += __popcll(m[k]);
        }
      } else {
#pragma unroll
        for (int k = 0; k < U; ++k) {
          const uint64_t pos = at + mbcnt(m[k]);
          if (((m[k] >> lane_id()) & 1u) && pos < capacity)
            reinterpret_cast<uint2*>(A.out)[pos] = make_uint2(uint32_t(b[k]), uint32_t(p[k]));
          at += uint64_t(__popcll(m[k]));
        }
      }
    };
    auto base_of = [&](uint32_t slot) {
      const uint64_t b = s_base[slot];
      return uint64_t(sgpr(uint32_t(b))) | (uint64_t(sgpr(uint32_t(b >> 32))) << 32);
    };
    for (uint32_t r0 = w.slo; r0 < w.shi; r0 += ROUND) {
      const bool more = r0 + ROUND < w.shi;
      if (more) load_probe(r0 + ROUND, w.shi, nk, np);
      const uint32_t nlane = opaque_tid();
      uint32_t bd[U], slow = 0, extra = 0;  // slow: probes that walk their bucket
      uint64_t m[U];
      int32_t fb[U];
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const uint32_t b = bounds_of(wide_hash(pk[k]));
        bd[k] = r0 + uint32_t(k) * BLOCK + nlane < w.shi ? b : 0u;
      }
#pragma unroll
      for (int k = 0; k < U; ++k) {
        const uint32_t lo = bd[k] & 0xFFFFu, n = (bd[k] >> 16) - lo;
        const uint32_t* tw = reinterpret_cast<const uint32_t*>(s_tag + (lo & ~3u));
        const uint32_t four = __builtin_amdgcn_alignbyte(tw[1], tw[0], lo);  // the tags of entries lo .. lo + 3
        const uint32_t t = wide_hash(pk[k]) << (bits + LGB);
        uint32_t z = zero_bytes(four ^ __builtin_amdgcn_perm(t, t, 0x03030303u));
        z &= n < 4u ? (1u << (8u * n)) - 1u : 0xFFFFFFFFu;
        // the first tag that fits; none: entry lo, unused
        fb[k] = int32_t(lo + (uint32_t(__builtin_ctz(z | 0x80000000u)) >> 3));
        bool hit = z != 0;
        const bool again = (n > 4u) | ((z & (z - 1u)) != 0);
        slow |= again & !(first_only & !VERIFY & hit) ? 1u << k : 0u;
        m[k] = __ballot(hit);
      }
      if constexpr (VERIFY) {
#pragma unroll
        for (int k = 0; k < U; ++k) {
          const bool hit = (m[k] >> lane_id()) & 1u;
          const bool same = hit & (s_key[fb[k]] == pk[k]);
          // another tag may still fit, or the bucket go on past the window
          if (first_only && same) slow &= ~(1u << k);
          m[k] = __ballot(same);
        }
      }
      if (__ballot(slow != 0)) {
#pragma unroll
        for (int k = 0; k < U; ++k) {
          bool hit = (m[k] >> lane_id()) & 1u;
          if (slow & (1u << k)) {
            uint32_t cnt = 0;
            const uint32_t h = wide_hash(pk[k]);
            for (uint32_t i = bd[k] & 0xFFFFu; i < bd[k] >> 16; ++i)
              if (entry_is(i, pk[k], h)) {
                if (cnt == 0) fb[k] = int32_t(i);
                ++cnt;
                if (first_only) break;
              }
            hit = cnt != 0;
            extra += cnt > 1u ? cnt - 1u : 0u;
          }
          m[k] = __ballot(hit);
        }
      }
      uint32_t wtot = 0;
#pragma unroll
      for (int k = 0; k < U; ++k) {
        fb[k] = s_pay[fb[k]];  // of the lanes that match; the others read some entry or spare bytes
        wtot += uint32_t(__popcll(m[k]));
      }
      const bool wave_multi = __ballot(extra != 0) != 0;
      uint32_t lane_pre = 0;  // multi-match rounds: the pairs of the lanes before this one
      if (wave_multi) {
        // a lane's count is below 2^21 (U probes of at most CAP matches), a wave's below 2^27
        uint32_t mine = extra;
#pragma unroll
        for (int k = 0; k < U; ++k) mine += uint32_t(m[k] >> lane_id()) & 1u;
        const uint32_t inc = wave_scan(mine);
        lane_pre = inc - mine;
        wtot = uint32_t(__builtin_amdgcn_readlane(int(inc), kWave - 1));
      }
      if (lane_id() == 0) s_wtot[par][wave] = wtot | (wave_multi ? 0x80000000u : 0u);
      if (threadIdx.x == 0) {
        if (pending) s_base[par ^ 1] = claim;
        if (!COLS && !more) s_next = ticket;
      }
      lds_barrier();
      // every wave's pairs, in the lanes of each wave
      const uint32_t wt = lane_id() < uint32_t(NW) ? s_wtot[par][lane_id()] : 0u;
      const bool any = __ballot(wt >> 31) != 0;
      const uint32_t wscan = wave_scan(wt & 0x7FFFFFFFu);  // below 2^32: 16 waves of less than 2^27
      const uint32_t pre = wave ? uint32_t(__builtin_amdgcn_readlane(int(wscan), int(wave) - 1)) : 0u;
      const uint32_t all = uint32_t(__builtin_amdgcn_readlane(int(wscan), NW - 1));
      // the next round's loads are waited for here, before any store is issued
      if (more) {
#pragma unroll
        for (int k = 0; k < U; ++k) {
          pin(nk[k]);
          pin(np[k]);
        }
      }
      if (threadIdx.x == 0 && all) claim = atomicAdd(A.d_count, (unsigned long long)all);
      if (pending) store_rows(base_of(par ^ 1) + h_pre, h_n, h_m, h_b, h_p);
      if (any) {
        // some probe matches more than once: claim now and walk again
        if (threadIdx.x == 0) s_base[par] = claim;
        lds_barrier();
        uint64_t at = base_of(par) + pre;
        if (wave_multi) {
          at += lane_pre;
#pragma unroll
          for (int k = 0; k < U; ++k)
            if ((m[k] >> lane_id()) & 1u) {
              const uint32_t h = wide_hash(pk[k]), b = bounds_of(h);
              for (uint32_t i = b & 0xFFFFu; i < b >> 16; ++i)
                if (entry_is(i, pk[k], h)) {
                  if (at < capacity) reinterpret_cast<uint2*>(A.out)[at] = make_uint2(uint32_t(s_pay[i]), uint32_t(pp[k]));
                  ++at;
                }
            }
        } else {
          store_rows(at, wtot, m, fb, pp);
        }
        pending = false;
      } else {
        pending = all != 0;
        h_pre = pre;
        h_n = wtot;
#pragma unroll
        for (int k = 0; k < U; ++k) {
          h_m[k] = m[k];
          h_b[k] = fb[k];
          h_p[k] = pp[k];
        }
      }
      par ^= 1;
      if (more) {
#pragma unroll
        for (int k = 0; k < U; ++k) {
          pk[k] = nk[k];
          pp[k] = np[k];
        }
      }
    }
    // ---- the next item's tuples are on their way while the last matches go out
    const uint32_t item_n = COLS ? item + grid : sgpr(s_next);
    const bool last = item_n >= total_items;
    if (!last) {
      w = decode(item_n);
      touch_build(w);
    }
    if (threadIdx.x == 0 && pending) s_base[par ^ 1] = claim;
    lds_barrier();  // also: every wave is done with the table
    if (pending) store_rows(base_of(par ^ 1) + h_pre, h_n, h_m, h_b, h_p);
    if (last) break;
    item = item_n;
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Shapes and launches
// ---------------------------------------------------------------------------
// Join configurations: {threads, build tuples per thread, log2 buckets, keys
// compared}.  The workgroups of the first two or three share a CU; the last
// fill its LDS alone.
struct WideCfg {
  int block, nb, lgb;
  bool verify;
  constexpr uint32_t cap() const { return uint32_t(block * nb); }
  constexpr size_t lds(int kb) const {
    return size_t(cap() + kWideSpare) * ((verify ? kb : 0) + 5) + (size_t(1) << lgb) * 2 + 8;
  }
};
static constexpr WideCfg kWideCfg4[5] = {{512, 6, 11, true}, {512, 12, 13, true}, {512, 17, 13, false},
                                         {1024, 17, 14, false}, {1024, 12, 14, true}};
static constexpr WideCfg kWideCfg8[3] = {{512, 4, 11, true}, {512, 10, 12, true}, {1024, 10, 13, true}};
static_assert(kWideCfg4[1].lds(4) <= 78 * 1024 && kWideCfg4[2].lds(4) <= 78 * 1024 && kWideCfg8[1].lds(8) <= 78 * 1024,
              "two workgroups per CU");
static_assert(kWideCfg4[3].lds(4) <= 158 * 1024 && kWideCfg4[4].lds(4) <= 158 * 1024 && kWideCfg8[2].lds(8) <= 158 * 1024,
              "LDS of one CU");

template <int KB, int CFG>
static hipError_t wide_join_t(const WideArgs& A, uint32_t grid, hipStream_t s) {
  constexpr WideCfg C = KB == 4 ? kWideCfg4[CFG] : kWideCfg8[KB == 4 ? 0 : CFG];
  constexpr int U = KB == 4 ? 8 : 6;
  if (A.bits == 0) {
    if constexpr (C.verify)
      hipLaunchKernelGGL((k_wide_join<KB, C.block, C.nb, U, C.lgb, C.verify, true>), dim3(grid), dim3(C.block), C.lds(KB), s, A);
  } else if constexpr (KB == 8 || CFG != 4) {
    hipLaunchKernelGGL((k_wide_join<KB, C.block, C.nb, U, C.lgb, C.verify, false>), dim3(grid), dim3(C.block), C.lds(KB), s, A);
  }
  return hipGetLastError();
}

static hipError_t wide_join(const WideArgs& A, int key_bytes, int cfg, hipStream_t s) {
  // persistent workgroups, as many as fit the 256 CUs at once; no more than
  // there can be items
  uint64_t most = uint64_t(1u << A.bits) + A.n[1] / A.slice + 1;
  if (A.bits == 0) most = (A.n[1] - 1) / A.slice + 1;
  const uint32_t fit = (key_bytes == 4 ? kWideCfg4[cfg] : kWideCfg8[cfg]).block == 1024 ? 256u : 512u;
  const uint32_t grid = most < fit ? uint32_t(most) : fit;
  if (key_bytes == 4) {
    switch (cfg) {
      case 0: return wide_join_t<4, 0>(A, grid, s);
      case 1: return wide_join_t<4, 1>(A, grid, s);
      case 2: return wide_join_t<4, 2>(A, grid, s);
      case 3: return wide_join_t<4, 3>(A, grid, s);
      default: return wide_join_t<4, 4>(A, grid, s);
    }
  }
  switch (cfg) {
    case 0: return wide_join_t<8, 0>(A, grid, s);
    case 1: return wide_join_t<8, 1>(A, grid, s);
    default: return wide_join_t<8, 2>(A, grid, s);
  }
}

bool wide_shape(int64_t nR, int64_t nS, int key_bytes, WideShape* W) {
  const double n = double(nR);
  auto cap = [&](int cfg) { return (key_bytes == 4 ? kWideCfg4[cfg] : kWideCfg8[cfg]).cap(); };
  // A scatter over 2048 digits costs less than one over 4096 (its runs are
  // twice as long), so the large chunks come before the last doubling of the
  // partitions: 20M x 90M int32 with payloads, 2048 partitions and chunks of
  // 17408 in workgroups of a CU each: scatter 390 us, join 376; 4096 and
  // chunks of 8704, two workgroups to a CU: 477 and 380.  16M x 64M int64
  // (tuples of 16 bytes then): 437 + 516 against 520 + 475.
  int cfg, bits = 0;
  // 2^b partitions of at most `aim` build rows on average.  No partitions
  // while one chunk holds the table: 3072 x 12288 int32 20 us, 6144 x 24576
  // 21 us, and with 12288 x 49152 at 30 us the line is reached (12289 rows in
  // 64 partitions 29 us).  The larger chunk takes over where the partitions
  // double otherwise: 1M x 4M 87 us with chunks of 3072, one row more with
  // 6144 74; 8M x 32M 328 on both sides of the line where the keys leave the
  // table.  Past the last line the two-pass pipeline: 67.1M x 134M int32
  // 1.74 ms here, one row more 2.40 ms there; 39.8M x 79.7M int64 1.51 and
  // 2.55 ms.
  auto bits_for = [&](double aim, int least) {
    int b = least;
    while (n / double(1 << b) > aim) ++b;
    return b;
  };
  if (key_bytes == 4) {
    if (nR <= int64_t(cap(0))) cfg = 0;
    else if (nR <= int64_t(cap(1))) cfg = 1;
    else if (nR <= int64_t(cap(4))) cfg = 4;
    else if (n <= 2048.0 * 512) { cfg = 0; bits = bits_for(2048.0, 6); }
    else if (n < 4096.0 * 2048) { cfg = 1; bits = bits_for(4096.0, 9); }
    else if (n <= 8192.0 * 2048) { cfg = 2; bits = bits_for(8192.0, 11); }
    else { cfg = 3; bits = n <= 16384.0 * 2048 ? 11 : 12; }
    if (n > 16384.0 * 4096) return false;
  } else {
    if (nR <= int64_t(cap(0))) cfg = 0;
    else if (nR <= int64_t(cap(1))) cfg = 1;
    else if (nR <= int64_t(cap(2))) cfg = 2;
    else if (n <= 1536.0 * 512) { cfg = 0; bits = bits_for(1536.0, 6); }
    else if (n <= 4608.0 * 2048) { cfg = 1; bits = bits_for(4608.0, 9); }
    else { cfg = 2; bits = n <= 9728.0 * 2048 ? 11 : 12; }
    if (n > 9728.0 * 4096) return false;
  }
  W->bits = bits;
  W->cfg = cfg;
  W->cap = cap(cfg);
  // Probe slices: every slice builds its chunk's table again, so a slice has
  // eight times the average chunk's rows, unless the items would not fill the
  // chip (1024 of them).
  const uint32_t round = uint32_t((key_bytes == 4 ? kWideCfg4[cfg] : kWideCfg8[cfg]).block * (key_bytes == 4 ? 8 : 6));
  const double chunk = n / double(1 << bits);
  double sl = 8.0 * chunk, fill = double(nS) / 1024.0;
  if (sl > fill) sl = fill > chunk ? fill : chunk;
  // With enough partitions an ordinary one is one item.
  if (bits >= 10 && sl < 1.25 * double(nS) / double(1 << bits)) sl = 1.25 * double(nS) / double(1 << bits);
  uint64_t slice = (uint64_t(sl) + round - 1) / round * round;
  if (slice < round) slice = round;
  W->slice = uint32_t(slice < (1u << 20) ? slice : (1u << 20));
  // Scatter tiles: 16 rows a thread (8 of 12-byte tuples), fewer when the
  // tables have too few rows to give every CU a few tiles (a tile's digits
  // cost the same whatever its rows: 1M x 4M in tiles of 4K, 64M in 16K).
  const int64_t rows = nR + nS;
  const int big = key_bytes == 4 ? 16 : 8;
  W->rows_per_thread = rows >= int64_t(512) * kWideBlock * big ? big : rows >= int64_t(512) * kWideBlock * big / 2 ? big / 2 : big / 4;
  return true;
}

// Rows left free after each partition, so that partitions start an odd number
// of 128-byte lines apart on average: the open lines of evenly filled
// partitions are otherwise in the same sets of the L2 (scatter of 64M x 256M
// 1340 us without, 1223 with).
static uint32_t wide_pad(int64_t n, int key_bytes, int bits) {
  const uint32_t lines = uint32_t((uint64_t(n) >> bits) * wide_tuple_bytes(key_bytes) / 128);
  // 16 tuples are a line of 8-byte tuples; 32 are three lines of 12-byte ones
  if (key_bytes == 4) return (lines % 2 ? 4u : 5u) * 16;
  return (lines % 2 ? 2u : 1u) * 32;
}

size_t wide_ws_bytes(int64_t nR, int64_t nS, int key_bytes, const WideShape& W) {
  if (W.bits == 0) return 0;
  auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
  const size_t P = size_t(1) << W.bits, tb = wide_tuple_bytes(key_bytes);
  const size_t scan = (P + kWideScan - 1) / kWideScan * kWideScan;
  return up((size_t(nR) + P * wide_pad(nR, key_bytes, W.bits)) * tb) +
         up((size_t(nS) + P * wide_pad(nS, key_bytes, W.bits)) * tb) + 2 * up(P * 4) + up(scan * 4) + up((3 * kWideScanMax + 1) * 4) +
         up(2 * kNumXcd * P * 4);
}

void wide_carve(int64_t nR, int64_t nS, int key_bytes, const WideShape& W, char* ws, char* end, WideArgs* A) {
  A->n[0] = uint32_t(nR);
  A->n[1] = uint32_t(nS);
  A->bits = W.bits;
  A->cap = W.cap;
  A->slice = W.slice;
  A->tile = uint32_t(W.rows_per_thread) * kWideBlock;
  if (W.bits == 0) return;
  auto take = [&](size_t b) {
    char* p = ws;
    ws += (b + 255) & ~size_t(255);
    return p;
  };
  const size_t P = size_t(1) << W.bits, tb = wide_tuple_bytes(key_bytes);
  A->pad[0] = wide_pad(nR, key_bytes, W.bits);
  A->pad[1] = wide_pad(nS, key_bytes, W.bits);
  A->tup[0] = take((size_t(nR) + P * A->pad[0]) * tb);
  A->tup[1] = take((size_t(nS) + P * A->pad[1]) * tb);
  A->start[0] = reinterpret_cast<uint32_t*>(take(P * 4));
  A->start[1] = reinterpret_cast<uint32_t*>(take(P * 4));
  A->iscan = reinterpret_cast<uint32_t*>(take((P + kWideScan - 1) / kWideScan * kWideScan * 4));
  A->bsum = reinterpret_cast<uint32_t*>(take((3 * kWideScanMax + 1) * 4));
  A->cnt = reinterpret_cast<uint32_t*>(end - ((2 * kNumXcd * P * 4 + 255) & ~size_t(255)));  // the workspace's last bytes
}

static bool aligned16w(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

hipError_t launch_wide_hist(const WideArgs& A, int key_bytes, hipStream_t s) {
  const uint32_t P = 1u << A.bits;
  hipError_t e = launch_fill_u64(reinterpret_cast<uint64_t*>(A.cnt), 0, int64_t(kNumXcd) * P, s);  // 2 tables x 4 bytes
  if (e != hipSuccess) return e;
  // two workgroups per CU, split between the tables by their sizes in multiples of 8
  const double share = double(A.n[0]) / (double(A.n[0]) + double(A.n[1]));
  int x0 = int(std::lround(share * 64.0));
  x0 = x0 < 1 ? 1 : x0 > 63 ? 63 : x0;
  const uint32_t g0 = uint32_t(x0) * kNumXcd;
  const bool vec = aligned16w(A.keys[0]) && aligned16w(A.keys[1]);
  const dim3 grid(64 * kNumXcd), block(kWideBlock);
#define PJ_WH(KB_, V_) hipLaunchKernelGGL((k_wide_hist<KB_, V_>), grid, block, P * 4, s, A, g0)
  if (key_bytes == 4) { if (vec) PJ_WH(4, true); else PJ_WH(4, false); }
  else { if (vec) PJ_WH(8, true); else PJ_WH(8, false); }
#undef PJ_WH
  return hipGetLastError();
}

hipError_t launch_wide_scan(const WideArgs& A, hipStream_t s) {
  const uint32_t P = 1u << A.bits;
  hipLaunchKernelGGL(k_wide_scan, dim3((P + kWideScan - 1) / kWideScan), dim3(kWideScan), 0, s, A);
  return hipGetLastError();
}

template <int KB, int E>
static hipError_t wide_scatter_t(const WideArgs& A, hipStream_t s) {
  const uint32_t P = 1u << A.bits, tile = kWideBlock * E;
  const size_t lds = size_t(tile) * wide_tuple_bytes(KB) + size_t(P) * 6 + 8;
  const uint32_t nt = (A.n[0] + tile - 1) / tile + kNumXcd + (A.n[1] + tile - 1) / tile;
  uint32_t grid = lds * 2 <= 150 * 1024 ? 512u : 256u;
  if (nt < grid) grid = (nt + kNumXcd - 1) / kNumXcd * kNumXcd;
  if (A.pay[0] || A.pay[1])
    hipLaunchKernelGGL((k_wide_scatter<KB, E, true>), dim3(grid), dim3(kWideBlock), lds, s, A);
  else
    hipLaunchKernelGGL((k_wide_scatter<KB, E, false>), dim3(grid), dim3(kWideBlock), lds, s, A);
  return hipGetLastError();
}

hipError_t launch_wide_scatter(const WideArgs& A, int key_bytes, hipStream_t s) {
  const int e = int(A.tile / kWideBlock);
  if (key_bytes == 4) return e == 16 ? wide_scatter_t<4, 16>(A, s) : e == 8 ? wide_scatter_t<4, 8>(A, s) : wide_scatter_t<4, 4>(A, s);
  return e == 8 ? wide_scatter_t<8, 8>(A, s) : e == 4 ? wide_scatter_t<8, 4>(A, s) : wide_scatter_t<8, 2>(A, s);
}

hipError_t launch_wide_join(const WideArgs& A, int key_bytes, int cfg, hipStream_t s) {
  if (A.bits == 0) {
    hipError_t e = launch_fill_u64(reinterpret_cast<uint64_t*>(A.d_count), 0, 1, s);
    if (e != hipSuccess) return e;
  }
  return wide_join(A, key_bytes, cfg, s);
}

}  // namespace pj
