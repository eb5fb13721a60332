// bucket_dev.hpp -- device code shared by the bucket sort (bucket.hip) and the
// sample sort (sample.hip): the key-width parameters, key helpers and the LDS
// radix passes.  Internal.
#pragma once

#include "kernels.hpp"
#include "tilescan.hpp"

namespace pgvd {

// ---- per key width ---------------------------------------------------------
// CAP keys (and labels) of one LDS sort item; BS threads of IPT keys each;
// scatter tiles of kBlock threads x TIPT keys.
template <typename K> struct Bk;
template <> struct Bk<uint32_t> { static constexpr int CAP = 8192, BS = 1024, IPT = 8, TIPT = 16; };
template <> struct Bk<uint64_t> { static constexpr int CAP = 5120, BS = 1024, IPT = 5, TIPT = 16; };
template <> struct Bk<Key128> { static constexpr int CAP = 2560, BS = 512, IPT = 5, TIPT = 8; };
// 64-bit halves of a key (OR / AND accumulation)
__device__ inline uint64_t klo(uint32_t a) { return a; }
__device__ inline uint64_t klo(uint64_t a) { return a; }
__device__ inline uint64_t klo(Key128 a) { return a.lo; }
__device__ inline uint64_t khi(uint32_t) { return 0; }
__device__ inline uint64_t khi(uint64_t) { return 0; }
__device__ inline uint64_t khi(Key128 a) { return a.hi; }

__device__ inline bool kless(uint32_t a, uint32_t b) { return a < b; }
__device__ inline bool kless(uint64_t a, uint64_t b) { return a < b; }
__device__ inline bool kless(Key128 a, Key128 b) { return a.hi < b.hi || (a.hi == b.hi && a.lo < b.lo); }

// nbits (<= 14) bits of a key from bit `shift` up
template <typename K>
__device__ inline uint32_t kbits(K a, int shift, uint32_t mask) {
  return klow32(kshr(a, shift)) & mask;
}

// all-ones key
template <typename K> __device__ inline K kones();
template <> __device__ inline uint32_t kones<uint32_t>() { return ~0u; }
template <> __device__ inline uint64_t kones<uint64_t>() { return ~0ull; }
template <> __device__ inline Key128 kones<Key128>() { return {~0ull, ~0ull}; }

// number of low bits that vary: bitlen(or ^ and)
__device__ inline int varying_bits(uint64_t olo, uint64_t ohi, uint64_t alo, uint64_t ahi) {
  const uint64_t xh = ohi ^ ahi, xl = olo ^ alo;
  return xh ? 128 - __builtin_clzll(xh) : (xl ? 64 - __builtin_clzll(xl) : 0);
}

// ---- LDS radix passes -------------------------------------------------------------
// Stable LSD passes in LDS over the BS IPT keys k[] (and labels v[]) of a
// workgroup; key index le = 64 IPT w + 64 j + lane lives in wave w,
// register j; ranks by ballot matching.  On return s_keys / s_vals hold the
// pairs in order of bits [0, 8 (passes - 1) + last_bits).  Slots past the
// item hold all-ones keys at the highest indices, which stay behind every
// real key.  s_cnt: NW 256 words, s_dig 256, s_w NW.
template <typename K, bool LAB, int BS, int IPT>
__device__ inline void lds_radix(K (&k)[IPT], uint32_t (&v)[IPT], int passes, int last_bits,
                                 K *s_keys, uint32_t *s_vals, uint32_t *s_cnt, uint32_t *s_dig,
                                 uint32_t *s_w) {
  constexpr int NW = BS / 64;
  static_assert(64 * IPT < (1 << 16), "a rank fits 16 bits");
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const uint32_t wofs = (uint32_t)w * 64u * IPT;
  for (int p = 0; p < passes; ++p) {
    const int sh = 8 * p;
    const int nbits = p == passes - 1 ? last_bits : 8;   // uniform
    const uint32_t dmask = (1u << nbits) - 1;
    for (int i = t; i < NW * 256; i += BS) s_cnt[i] = 0;
    __syncthreads();
    uint32_t rk[IPT];   // rank within (wave, digit) | digit << 16
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const uint32_t d = kdigit(k[j], sh) & dmask;
      uint32_t plo = ~0u, phi = ~0u;
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        if (b < nbits) {
          const int32_t sb = __builtin_amdgcn_sbfe((int32_t)d, b, 1);
          const uint64_t bb = __ballot(sb < 0);
          plo = __builtin_amdgcn_bitop3_b32(plo, (uint32_t)bb, (uint32_t)sb, 0x90);
          phi = __builtin_amdgcn_bitop3_b32(phi, (uint32_t)(bb >> 32), (uint32_t)sb, 0x90);
        }
      }
      const uint32_t c = s_cnt[w * 256 + d];
      const uint32_t below = __builtin_amdgcn_mbcnt_hi(phi, __builtin_amdgcn_mbcnt_lo(plo, 0u));
      rk[j] = (c + below) | (d << 16);
      // every lane of the group stores the same new count
      s_cnt[w * 256 + d] = c + (uint32_t)(__popc(plo) + __popc(phi));
    }
    __syncthreads();
    uint32_t tot = 0;
    if (t < 256) {
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) {
        const uint32_t c = s_cnt[ww * 256 + t];
        s_cnt[ww * 256 + t] = tot;
        tot += c;
      }
    }
    uint32_t all;
    const uint32_t dex = block_excl_sum<uint32_t, NW>(tot, s_w, &all);
    if (t < 256) s_dig[t] = dex;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const uint32_t d = rk[j] >> 16;
      const uint32_t q = (rk[j] & 0xffffu) + s_dig[d] + s_cnt[w * 256 + d];
      s_keys[q] = k[j];
      if (LAB) s_vals[q] = v[j];
    }
    __syncthreads();
    if (p + 1 < passes) {
#pragma unroll
      for (int j = 0; j < IPT; ++j) {
        k[j] = s_keys[wofs + j * 64 + lane];
        if (LAB) v[j] = s_vals[wofs + j * 64 + lane];
      }
      __syncthreads();   // s_keys and s_cnt are rewritten by the next pass
    }
  }
}

// ---- merge sort of one item in LDS -----------------------------------------------
// (key, position) pairs in a strict total order: equal keys by position, so
// the sort is stable and slots past the item (all-ones keys, positions >=
// cnt) stay behind every real key.
template <typename K>
__device__ inline bool pair_lt(const K &a, uint32_t ia, const K &b, uint32_t ib) {
  return kless(a, b) || (keq(a, b) && ia < ib);
}

// The cnt keys pick(i) (and labels vpick(i)) sorted by merging: each
// thread sorts IPT consecutive keys in registers, then log2(BS) rounds merge
// runs pairwise, every thread producing IPT outputs of its run pair from a
// merge-path split found by binary search.  The cost does not depend on how
// the keys are spread, which suits wide keys that no few digits separate
// (sparse 128-bit keys on curves).  Positions travel in s_idx (16 bits);
// labels, staged in s_vals in input order, are gathered by position at the
// end.  On return s_keys[0 .. cnt) (and s_vals) hold the item in order.
template <typename K, bool LAB, int BS, int IPT, typename Pick, typename VPick>
__device__ inline void lds_merge_sort(Pick pick, VPick vpick, uint32_t cnt, K *s_keys,
                                      uint32_t *s_vals, uint16_t *s_idx) {
  constexpr uint32_t CAP = (uint32_t)BS * IPT;
  static_assert(CAP <= 65536, "positions fit 16 bits");
  const uint32_t t = threadIdx.x;
  const uint32_t p0 = t * IPT;
  K k[IPT];
  uint32_t x[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t p = p0 + j;
    k[j] = p < cnt ? pick(p) : kones<K>();
    x[j] = p;
    if (LAB && p < cnt) s_vals[p] = vpick(p);
  }
  // odd-even transposition sort of the thread's IPT pairs
#pragma unroll
  for (int r = 0; r < IPT; ++r) {
#pragma unroll
    for (int j = r & 1; j + 1 < IPT; j += 2) {
      if (pair_lt(k[j + 1], x[j + 1], k[j], x[j])) {
        const K tk = k[j]; k[j] = k[j + 1]; k[j + 1] = tk;
        const uint32_t tx = x[j]; x[j] = x[j + 1]; x[j + 1] = tx;
      }
    }
  }
  for (uint32_t w = IPT; w < CAP && w < cnt; w *= 2) {   // (past cnt: nothing but the slots after it)
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      s_keys[p0 + j] = k[j];
      s_idx[p0 + j] = (uint16_t)x[j];
    }
    __syncthreads();
    const uint32_t base = p0 / (2 * w) * (2 * w);
    const uint32_t d = p0 - base;   // this thread's first output in the merged pair
    const uint32_t A = base, B = base + w;
    // i keys from run A and d - i from run B come first
    uint32_t lo = d > w ? d - w : 0u, hi = d < w ? d : w;
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      const uint32_t bj = B + d - 1 - mid;
      if (pair_lt(s_keys[bj], (uint32_t)s_idx[bj], s_keys[A + mid], (uint32_t)s_idx[A + mid]))
        hi = mid;
      else
        lo = mid + 1;
    }
    uint32_t ai = A + lo, bi = B + (d - lo);
    const uint32_t ae = A + w, be = B + w;
    K ka = ai < ae ? s_keys[ai] : kones<K>(), kb = bi < be ? s_keys[bi] : kones<K>();
    uint32_t xa = ai < ae ? s_idx[ai] : 0xffffffffu, xb = bi < be ? s_idx[bi] : 0xffffffffu;
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      const bool take_a = pair_lt(ka, xa, kb, xb);   // an exhausted run compares last
      k[j] = take_a ? ka : kb;
      x[j] = take_a ? xa : xb;
      if (take_a) {
        ++ai;
        ka = ai < ae ? s_keys[ai] : kones<K>();
        xa = ai < ae ? s_idx[ai] : 0xffffffffu;
      } else {
        ++bi;
        kb = bi < be ? s_keys[bi] : kones<K>();
        xb = bi < be ? s_idx[bi] : 0xffffffffu;
      }
    }
    __syncthreads();   // every read of this round is done before the next writes
  }
  uint32_t lab[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) lab[j] = (LAB && x[j] < cnt) ? s_vals[x[j]] : 0u;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    s_keys[p0 + j] = k[j];
    if (LAB) s_vals[p0 + j] = lab[j];
  }
}

// ---- minimum and maximum, differences of keys -------------------------------------
__device__ inline uint32_t ksub(uint32_t a, uint32_t b) { return a - b; }
__device__ inline uint64_t ksub(uint64_t a, uint64_t b) { return a - b; }
__device__ inline Key128 ksub(Key128 a, Key128 b) {
  return {a.lo - b.lo, a.hi - b.hi - (a.lo < b.lo ? 1ull : 0ull)};
}
// The smaller and the larger key (by value: a conditional on two structs picks
// an address and sends both to scratch memory).
template <typename K> __device__ inline K kmin(K a, K b) { return kless(a, b) ? a : b; }
template <typename K> __device__ inline K kmax(K a, K b) { return kless(a, b) ? b : a; }
template <> __device__ inline Key128 kmin<Key128>(Key128 a, Key128 b) {
  const bool l = kless(a, b);
  return {l ? a.lo : b.lo, l ? a.hi : b.hi};
}
template <> __device__ inline Key128 kmax<Key128>(Key128 a, Key128 b) {
  const bool l = kless(a, b);
  return {l ? b.lo : a.lo, l ? b.hi : a.hi};
}
__device__ inline uint32_t kshfl_xor(uint32_t a, int d) { return (uint32_t)__shfl_xor((int)a, d, 64); }
__device__ inline uint64_t kshfl_xor(uint64_t a, int d) {
  return (uint64_t)__shfl_xor((unsigned long long)a, d, 64);
}
__device__ inline Key128 kshfl_xor(Key128 a, int d) {
  return {kshfl_xor(a.lo, d), kshfl_xor(a.hi, d)};
}

// Smallest and largest key over the workgroup of BS threads, of each
// thread's own (mn, mx); s_mm holds 2 BS / 64 keys.  Passes one barrier;
// s_mm is free after the caller's next one.
template <typename K, int BS>
__device__ inline void block_minmax(K &mn, K &mx, K *s_mm) {
  constexpr int NW = BS / 64;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    mn = kmin(mn, kshfl_xor(mn, d));
    mx = kmax(mx, kshfl_xor(mx, d));
  }
  if ((threadIdx.x & 63) == 0) {
    s_mm[threadIdx.x >> 6] = mn;
    s_mm[NW + (threadIdx.x >> 6)] = mx;
  }
  __syncthreads();
  for (int w = 0; w < NW; ++w) {
    mn = kmin(mn, s_mm[w]);
    mx = kmax(mx, s_mm[NW + w]);
  }
}

// The last steps of an LDS sort whose keys sit, in bucket order, in s_keys:
// each key's rank within its bucket [b0[j], b1[j]) by reading the others
// (four at a time; ties by slot at[j]), then one permutation.
template <typename K, bool LAB, int BS, int IPT>
__device__ inline void lds_rank(const K (&k)[IPT], const uint32_t (&v)[IPT], uint32_t cnt,
                                uint32_t (&at)[IPT], const uint32_t (&b0)[IPT],
                                const uint32_t (&b1)[IPT], K *s_keys, uint32_t *s_vals) {
  const uint32_t t = threadIdx.x;
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if ((uint32_t)j * BS + t < cnt) {
      uint32_t r = b0[j];
      for (uint32_t x = b0[j]; x < b1[j]; x += 4) {
        K y[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) y[u] = s_keys[min(x + u, b1[j] - 1)];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
          r += (x + u < b1[j] && (kless(y[u], k[j]) || (keq(y[u], k[j]) && x + u < at[j]))) ? 1u : 0u;
      }
      at[j] = r;
    }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if ((uint32_t)j * BS + t < cnt) {
      s_keys[at[j]] = k[j];
      if (LAB) s_vals[at[j]] = v[j];
    }
}

// ---- LDS sort by splitters -------------------------------------------------------
// Sorts the cnt <= BS IPT pairs (k[j], v[j]) at index i = j BS + threadIdx.x in
// LDS, whatever their distribution: 255 splitters, evenly spaced positions of
// the input ranked against each other, bound 256 buckets; every key finds its
// bucket (8 LDS reads), and its rank within the bucket by reading the others
// in it (cnt / 256 on average).  Keys compare together with their index, so
// equal keys spread over buckets like distinct ones.  pick(i) reads key i.  On
// return (no barrier passed since) s_keys / s_vals hold the pairs in order;
// s_tmp: split_words<K>() words, aligned as K.
constexpr int kSplits = 256;
template <typename K>
constexpr int split_words() { return kSplits * ((int)sizeof(K) / 4 + 3) + 1 + 16; }

template <typename K, bool LAB, int BS, int IPT, typename Pick>
__device__ inline void lds_split_sort(K (&k)[IPT], uint32_t (&v)[IPT], uint32_t cnt, Pick pick,
                                      K *s_keys, uint32_t *s_vals, uint32_t *s_tmp) {
  constexpr int NW = BS / 64, PARTS = BS / kSplits, PER = kSplits / PARTS;
  static_assert(BS % kSplits == 0 && NW <= 16, "every thread ranks against a part");
  K *s_sp = reinterpret_cast<K *>(s_tmp);              // splitters as picked, then in order
  uint32_t *s_pos = s_tmp + kSplits * (int)sizeof(K) / 4;   // their indexes, in order
  uint32_t *s_cnt = s_pos + kSplits;                   // their ranks, then the buckets' counts
  uint32_t *s_start = s_cnt + kSplits;                 // kSplits + 1
  uint32_t *s_w = s_start + kSplits + 1;
  const uint32_t t = threadIdx.x;
  const uint32_t pos = (t & (kSplits - 1)) * cnt / kSplits;
  K mine = kzero_value<K>();
  if (t < kSplits) {
    mine = pick(pos);
    s_sp[t] = mine;
    s_cnt[t] = 0;
  }
  __syncthreads();
  {
    const uint32_t j = t & (kSplits - 1), i0 = t / kSplits * PER;
    const K x = s_sp[j];
    uint32_t r = 0;
#pragma unroll 8
    for (uint32_t i = i0; i < i0 + PER; ++i) {
      const K y = s_sp[i];
      r += (kless(y, x) || (keq(y, x) && i < j)) ? 1u : 0u;
    }
    atomicAdd(&s_cnt[j], r);
  }
  __syncthreads();
  if (t < kSplits) {
    const uint32_t r = s_cnt[t];
    s_sp[r] = mine;
    s_pos[r] = pos;
    s_cnt[t] = 0;
  }
  __syncthreads();
  uint32_t lo[IPT], rs[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) lo[j] = 0;
  // (every key's search at once: their reads are independent)
#pragma unroll
  for (uint32_t step = kSplits / 2; step >= 1; step >>= 1) {
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
      if ((uint32_t)j * BS >= cnt) break;   // uniform
      const uint32_t at = lo[j] + step;
      const K y = s_sp[at];
      const bool le = kless(y, k[j]) || (keq(y, k[j]) && s_pos[at] <= (uint32_t)j * BS + t);
      lo[j] = le ? at : lo[j];
    }
  }
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    rs[j] = (uint32_t)j * BS + t < cnt ? atomicAdd(&s_cnt[lo[j]], 1u) : 0u;
  __syncthreads();
  uint32_t total;
  const uint32_t ex = block_excl_sum<uint32_t, NW>(t < kSplits ? s_cnt[t] : 0u, s_w, &total);
  if (t < kSplits) s_start[t] = ex;
  if (t == 0) s_start[kSplits] = total;
  __syncthreads();
  uint32_t b1[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if ((uint32_t)j * BS + t < cnt) {
      b1[j] = s_start[lo[j] + 1];
      lo[j] = s_start[lo[j]];
      rs[j] += lo[j];
      s_keys[rs[j]] = k[j];
    }
  __syncthreads();
  lds_rank<K, LAB, BS, IPT>(k, v, cnt, rs, lo, b1, s_keys, s_vals);
}

// ---- LDS sort by bins -------------------------------------------------------------
// Sorts in LDS the cnt <= BS IPT pairs (k[j], v[j]) at index i = j BS +
// threadIdx.x, for keys that are spread smoothly for the most part: counted in
// 4096 bins of their range (the keys less the smallest); where some bin holds
// more than kBinRank of them, every bin is cut into as many bins as it holds
// keys (rounded down to a power of two) and the keys are counted again; then
// each key is ranked within its bin.  A bin of more than RANK2 keys that are all
// the same (many points at one place) needs no ranking; keys too close together
// even for that (a range that spans two tight clusters) go to the merge sort
// (MERGE) or are ranked against splitters.  The merge sort is the better one for
// many keys a thread (8192 64-bit keys of 1024 threads 60 us, by splitters 117;
// the 512-thread sorts of a batch of 384 instances 487 and 507 us), the splitters
// for few (300,007 clustered points, 1024 threads a bucket: 33.6 and 29.7 us)
// and for 128-bit keys (2^22 labelled loop samples: 159 and 151 us), each with
// the RANK2 that suited it of 64 and 128; kBinRank 12, 24 and 48 time alike.
// pick(i) and vpick(i) read pair i again.  On return (no barrier passed since)
// s_keys / s_vals hold the pairs in order, equal keys in any order; s_tmp:
// bin_words<K, BS>() words, aligned as K.
constexpr int kBins = 4096;
constexpr uint32_t kBinRank = 24;
template <typename K, int BS>
constexpr int bin_words() {
  return kBins + 4 + 2 * (BS / 64) * ((int)sizeof(K) / 4) + 2 * (BS / 64);
}

// Largest v over the workgroup (two barriers); s_mx holds BS / 64 words.
template <int BS>
__device__ inline uint32_t block_max(uint32_t v, uint32_t *s_mx) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, d, 64));
  if ((threadIdx.x & 63) == 0) s_mx[threadIdx.x >> 6] = v;
  __syncthreads();
  for (int w = 0; w < BS / 64; ++w) v = max(v, s_mx[w]);
  __syncthreads();
  return v;
}

template <typename K, bool LAB, int BS, int IPT, bool MERGE, typename Pick, typename VPick>
__device__ inline void lds_bin_sort(K (&k)[IPT], uint32_t (&v)[IPT], uint32_t cnt, Pick pick,
                                    VPick vpick, K *s_keys, uint32_t *s_vals, uint32_t *s_tmp) {
  constexpr int NW = BS / 64, PER = kBins / BS;
  constexpr uint32_t RANK2 = MERGE ? 128 : 64;
  constexpr int kMid = kBins + 4;
  static_assert(2 * BS * IPT <= 4 * kMid && split_words<K>() <= kMid,
                "the other sorts' tables fit");
  uint32_t *s_bin = s_tmp;
  K *s_mm = reinterpret_cast<K *>(s_tmp + kMid);
  uint32_t *s_w = s_tmp + kMid + 2 * NW * ((int)sizeof(K) / 4), *s_mx = s_w + NW;
  const uint32_t t = threadIdx.x;
  K mn = kones<K>(), mx = kzero_value<K>();
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if ((uint32_t)j * BS + t < cnt) {
      mn = kmin(mn, k[j]);
      mx = kmax(mx, k[j]);
    }
  for (uint32_t i = t; i < (uint32_t)kBins; i += BS) s_bin[i] = 0;
  block_minmax<K, BS>(mn, mx, s_mm);
  const K span = ksub(mx, mn);
  const int eff = varying_bits(klo(span), khi(span), 0, 0);   // uniform
  const int shift = eff > 12 ? eff - 12 : 0;
  uint32_t bin[IPT], at[IPT], b0[IPT], b1[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    bin[j] = kbits(ksub(k[j], mn), shift, kBins - 1);
    at[j] = (uint32_t)j * BS + t < cnt ? atomicAdd(&s_bin[bin[j]], 1u) : 0u;
  }
  __syncthreads();
  uint32_t c[PER], run = 0, most = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    c[i] = s_bin[t * PER + i];
    run += c[i];
    most = max(most, c[i]);
  }
  most = block_max<BS>(most, s_mx);
  uint32_t total;
  if (most <= kBinRank || shift == 0) {   // (shift 0: a bin holds equal keys)
    uint32_t ex = block_excl_sum<uint32_t, NW>(run, s_w, &total);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      s_bin[t * PER + i] = ex;
      ex += c[i];
    }
    if (t == 0) s_bin[kBins] = total;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < IPT; ++j)
      if ((uint32_t)j * BS + t < cnt) {
        b0[j] = s_bin[bin[j]];
        b1[j] = s_bin[bin[j] + 1];
        at[j] += b0[j];
        s_keys[at[j]] = k[j];
        if (LAB && shift == 0) s_vals[at[j]] = v[j];
      }
    if (shift == 0) return;
    __syncthreads();
    lds_rank<K, LAB, BS, IPT>(k, v, cnt, at, b0, b1, s_keys, s_vals);
    return;
  }
  // the second counting: bin b's own bins start at entry off[b] of s_cnt2
  // (in the keys' space, not yet used): off | log2(bins) << 16
  uint32_t *s_cnt2 = reinterpret_cast<uint32_t *>(s_keys);
  static_assert(BS * IPT <= 65536, "an offset fits 16 bits");
  uint32_t sub = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i)
    if (c[i]) sub += 1u << min(31 - __clz((int)c[i]), shift);
  uint32_t n2;
  uint32_t off = block_excl_sum<uint32_t, NW>(sub, s_w, &n2);   // n2 <= cnt
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const uint32_t lg = c[i] ? (uint32_t)min(31 - __clz((int)c[i]), shift) : 0u;
    s_bin[t * PER + i] = off | lg << 16;
    off += c[i] ? 1u << lg : 0u;
  }
  for (uint32_t i = t; i < n2; i += BS) s_cnt2[i] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if ((uint32_t)j * BS + t < cnt) {
      const uint32_t e = s_bin[bin[j]], lg = e >> 16;
      bin[j] = (e & 0xffffu) + kbits(ksub(k[j], mn), shift - (int)lg, (1u << lg) - 1u);
      at[j] = atomicAdd(&s_cnt2[bin[j]], 1u);
    }
  __syncthreads();
  uint32_t c2[IPT];
  run = 0;
  most = 0;
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    c2[i] = t * IPT + i < n2 ? s_cnt2[t * IPT + i] : 0u;
    run += c2[i];
    most = max(most, c2[i]);
  }
  most = block_max<BS>(most, s_mx);
  uint32_t ex = block_excl_sum<uint32_t, NW>(run, s_w, &total);
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    if (t * IPT + i < n2) s_cnt2[t * IPT + i] = ex;
    ex += c2[i];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if ((uint32_t)j * BS + t < cnt) {
      b0[j] = s_cnt2[bin[j]];
      b1[j] = bin[j] + 1 < n2 ? s_cnt2[bin[j] + 1] : cnt;
      at[j] += b0[j];
    }
  __syncthreads();   // the counts are read: the keys take their space
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if ((uint32_t)j * BS + t < cnt) s_keys[at[j]] = k[j];
  __syncthreads();
  if (most > RANK2) {   // uniform
    // a crowded bin of one key's copies is in order as it is
    uint32_t mixed = 0;
#pragma unroll
    for (int j = 0; j < IPT; ++j)
      if ((uint32_t)j * BS + t < cnt && b1[j] - b0[j] > RANK2) {
        mixed |= keq(k[j], s_keys[b0[j]]) ? 0u : 1u;
        b0[j] = b1[j] = at[j];
      }
    if (block_max<BS>(mixed, s_mx)) {
      if constexpr (!MERGE)
        lds_split_sort<K, LAB, BS, IPT>(k, v, cnt, pick, s_keys, s_vals, s_tmp);
      else
        lds_merge_sort<K, LAB, BS, IPT>(pick, vpick, cnt, s_keys, s_vals,
                                        reinterpret_cast<uint16_t *>(s_tmp));
      return;
    }
  }
  lds_rank<K, LAB, BS, IPT>(k, v, cnt, at, b0, b1, s_keys, s_vals);
}

}  // namespace pgvd
