// sample.hip -- a sample sort of one or many segments of keys, for sets whose
// top key bits do not spread them (clusters): the batched form's sort, and
// the whole path's where the bucket sort's plan finds most keys crowded.
//
// Per segment of n keys, nb = n / T buckets (T well under the CAP keys that
// one LDS sort holds) are bounded by splitters taken from a sorted sample of
// 16 keys per bucket, so a bucket holds T keys on average whatever the
// distribution.  One pass counts the keys per bucket, one scatters them, and
// an LDS sort orders each bucket: keys are read three times and
// written twice, where eight radix passes read and write them eight times.
// A key that the sample holds twice gets a bucket of its own (its successor
// is a splitter too), so repeated keys do not swell a bucket of distinct
// ones.  A bucket above CAP is written from its one key by many workgroups
// (a repeated key) or sorted in global memory by one (a rare sample).
//
// Equal keys may come out in any order (their labels too), as from the bucket
// sort.  No count comes back to the host: the launches depend only on the
// segments' sizes, so a batch's graph holds them.
#include "bucket_dev.hpp"

namespace pgvd {

namespace {

// An LDS sort holds at most CAP keys (a multiple of 1024).
template <typename K> struct SsItem;
template <> struct SsItem<uint32_t> { static constexpr int CAP = 8192; };
template <> struct SsItem<uint64_t> { static constexpr int CAP = 5120; };
template <> struct SsItem<Key128> { static constexpr int CAP = 3072; };
constexpr int kSsBlock = 1024;        // threads of the sample's sort
constexpr int kSsIpt = 8;             // its keys per thread, at most
static_assert(kSsBlock * kSsIpt == 16 * kSsMaxBuckets, "16 sample keys per bucket");
// Splitters are looked up through a table of the key's top kSsLutBits bits:
// entry w is the number of splitters below window w, so a search only runs
// over the splitters of the key's own window.
constexpr int kSsLutBits = 12;
constexpr int kSsLut = (1 << kSsLutBits) + 1;
static_assert(kSsLutWords * 2 >= kSsLut, "the table's room in the workspace");

__device__ inline uint32_t ksucc(uint32_t a) { return a + 1; }
__device__ inline uint64_t ksucc(uint64_t a) { return a + 1; }
__device__ inline Key128 ksucc(Key128 a) {
  return {a.lo + 1, a.hi + (a.lo == ~0ull ? 1ull : 0ull)};
}

// Segment s of the plan (the single one without tables).
struct SsSeg {
  uint32_t kofs, n, bucket, nb;
};
__device__ inline SsSeg ss_segment(const SsPlan &p, uint32_t s) {
  if (!p.seg) return {0u, p.n, 0u, p.nb};
  return {p.seg[s].kofs, p.seg[s].n, p.bucket_first[s],
          p.bucket_first[s + 1] - p.bucket_first[s]};
}

// Where a segment's sorted keys go and its duplicates are reported.
struct SsOut {
  uint32_t kofs, prepend, shift;
  uint32_t *dups;
};
__device__ inline SsOut ss_out(const SsPlan &p, uint32_t s, uint32_t prepend, RunState *st) {
  if (!p.ss) return {0u, prepend, 0u, &st->msd_dups};
  const uint32_t pre = p.seg[s].prepend;
  return {p.seg[s].kofs, pre, pre, &p.ss[s].dups};
}

// Deterministic 32-bit mix (the sample's position within its stratum):
// "lowbias32", a published xor-shift-multiply hash whose constants a search by
// C. Wellons (hash-prospector) found.
__device__ inline uint32_t mix32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  x ^= x >> 16;
  return x;
}

// One workgroup per segment: the sample (one key from each of nb * 16 strata
// of the segment), sorted in LDS, gives splitters [1, nb); splitter 0 stands
// for the lowest key.
template <typename K, int IPT>
__global__ __launch_bounds__(kSsBlock) void ss_splitters_kernel(const K *__restrict__ keys,
                                                                SsPlan p, int mbits) {
  __shared__ K s_keys[kSsBlock * IPT];
  __shared__ __align__(16) uint32_t s_tmp[bin_words<K, kSsBlock>()];
  __shared__ K s_sp[kSsMaxBuckets];
  const uint32_t s = p.multi ? p.multi[blockIdx.x] : blockIdx.x;
  const SsSeg sg = ss_segment(p, s);
  const int t = threadIdx.x;
  const uint32_t S = sg.nb * 16;   // <= kSsBlock * IPT, and S <= n (a bucket averages above 16)
  // stratum i: keys [i n / S, (i + 1) n / S) in 16-bit fixed point; the key
  // within it by a hash
  const uint64_t step = ((uint64_t)sg.n << 16) / S;   // >= 2^16
  auto sample = [&](uint32_t i) {
    const uint32_t a = (uint32_t)((i * step) >> 16), b = (uint32_t)(((i + 1) * step) >> 16);
    return keys[sg.kofs + a + __umulhi(mix32(i * 0x9e3779b9u + s), b - a)];
  };
  K k[IPT];
  uint32_t v[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = (uint32_t)j * kSsBlock + t;
    k[j] = i < S ? sample(i) : kzero_value<K>();
    v[j] = 0;
  }
  lds_bin_sort<K, false, kSsBlock, IPT, (IPT > 4)>(
      k, v, S, sample, [](uint32_t) { return 0u; }, s_keys, nullptr, s_tmp);
  __syncthreads();
  // splitter j = sample 16 j; the second of a run of equal ones becomes the
  // run's successor, which closes the repeated key's own bucket
  for (uint32_t j = t; j < sg.nb; j += kSsBlock) {
    K x = j ? s_keys[j * 16] : kzero_value<K>();
    if (j >= 2 && keq(s_keys[j * 16], s_keys[(j - 1) * 16]) && !keq(x, kones<K>())) x = ksucc(x);
    s_sp[j] = x;
    static_cast<K *>(p.splitters)[sg.bucket + j] = x;
  }
  __syncthreads();
  const int shift = mbits > kSsLutBits ? mbits - kSsLutBits : 0;
  uint16_t *lut = reinterpret_cast<uint16_t *>(p.lut + (size_t)blockIdx.x * kSsLutWords);
  for (uint32_t x = t; x < (uint32_t)kSsLut; x += kSsBlock) {
    // splitters j in [1, nb) whose window is below x
    uint32_t lo = 0, hi = sg.nb - 1;
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (klow32(kshr(s_sp[mid], shift)) < x) lo = mid; else hi = mid - 1;
    }
    lut[x] = (uint16_t)lo;
  }
}

// Counts the keys of each tile per bucket and keeps every key's bucket (16
// bits) for the scatter.
template <typename K>
__global__ __launch_bounds__(kBlock) void ss_count_kernel(const K *__restrict__ keys, SsPlan p,
                                                          int mbits) {
  constexpr int IPT = Bk<K>::TIPT, TILE = kBlock * IPT;
  __shared__ uint32_t s_cnt[kSsMaxBuckets];
  __shared__ K s_sp[kSsMaxBuckets];
  __shared__ uint32_t s_lut[kSsLutWords];
  const uint32_t tile = blockIdx.x;
  if (p.limits && tile >= p.limits[0]) return;
  const uint32_t s = p.seg ? p.tiles.seg[tile] : 0u;
  const SsSeg sg = ss_segment(p, s);
  const int t = threadIdx.x;
  const uint32_t lo0 = (tile - (p.seg ? p.tiles.first[s] : 0u)) * (uint32_t)TILE;
  const uint32_t hi0 = min(lo0 + (uint32_t)TILE, sg.n);
  K k[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = lo0 + j * kBlock + t;
    k[j] = keys[sg.kofs + (i < hi0 ? i : lo0)];
  }
  const K *sp = static_cast<const K *>(p.splitters) + sg.bucket;
  for (uint32_t j = t; j < sg.nb; j += kBlock) {
    s_cnt[j] = 0;
    s_sp[j] = sp[j];
  }
  const uint32_t *lut = p.lut + (size_t)(p.multi_of ? p.multi_of[s] : s) * kSsLutWords;
  for (uint32_t j = t; j < (uint32_t)kSsLutWords; j += kBlock) s_lut[j] = lut[j];
  __syncthreads();
  const uint16_t *s_l = reinterpret_cast<const uint16_t *>(s_lut);
  const int shift = mbits > kSsLutBits ? mbits - kSsLutBits : 0;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = lo0 + j * kBlock + t;
    const uint32_t x = klow32(kshr(k[j], shift)) & ((1u << kSsLutBits) - 1);
    uint32_t lo = s_l[x], hi = s_l[x + 1];
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (kless(k[j], s_sp[mid])) hi = mid - 1; else lo = mid;
    }
    if (i < hi0) {
      atomicAdd(&s_cnt[lo], 1u);
      p.ids[sg.kofs + i] = (uint16_t)lo;
    }
  }
  __syncthreads();
  for (uint32_t j = t; j < sg.nb; j += kBlock)
    if (s_cnt[j]) atomicAdd(&p.counts[sg.bucket + j], s_cnt[j]);
}

constexpr unsigned kSsBigGrid = 256;
// How ss_big_kernel treats an item: as keys to sort, or as a run of one key.
constexpr uint32_t kSsBigSort = 1, kSsBigRun = 2;

// Bucket b holds copies of its splitter alone: the next splitter is its
// successor (ss_splitters_kernel closes a repeated key's bucket so), or it is
// the largest key there is.
template <typename K>
__device__ inline bool ss_one_key(const K *sp, uint32_t b, uint32_t nb, int mbits) {
  const K x = sp[b];
  if (b + 1 < nb) return keq(sp[b + 1], ksucc(x));
  return keq(x, kshr(kones<K>(), (int)sizeof(K) * 8 - mbits));
}

// One workgroup per segment: bucket starts from the counts, as the scatter's
// cursors and the LDS sort's items; buckets above CAP are listed for
// ss_big_kernel, one key's copies in runs of up to CAP.
template <typename K>
__global__ __launch_bounds__(kSsMaxBuckets) void ss_plan_kernel(SsPlan p, uint32_t cap, int mbits,
                                                                RunState *st) {
  __shared__ uint32_t s_w[kSsMaxBuckets / 64];
  const uint32_t s = p.multi ? p.multi[blockIdx.x] : blockIdx.x;
  const SsSeg sg = ss_segment(p, s);
  const uint32_t b = threadIdx.x;
  const uint32_t c = b < sg.nb ? p.counts[sg.bucket + b] : 0u;
  uint32_t total;
  const uint32_t at = sg.kofs + block_excl_sum<uint32_t, kSsMaxBuckets / 64>(c, s_w, &total);
  if (b < sg.nb) {
    p.cursors[sg.bucket + b] = at;
    BkItem it{at, c, 1u, s};   // (sbits: the segment)
    if (c > cap) {
      if (ss_one_key(static_cast<const K *>(p.splitters) + sg.bucket, b, sg.nb, mbits)) {
        constexpr uint32_t RUN = (uint32_t)SsItem<K>::CAP;
        const uint32_t runs = (c + RUN - 1) / RUN, first = atomicAdd(p.n_big, runs);
        for (uint32_t r = 0; r < runs; ++r)
          p.big[first + r] = {at + r * RUN, min(RUN, c - r * RUN), kSsBigRun, s};
      } else {
        p.big[atomicAdd(p.n_big, 1u)] = {at, c, kSsBigSort, s};
      }
      it.count = 0;
    }
    p.items[sg.bucket + b] = it;
  }
  if (!p.seg && b == 0) {   // the whole path's keys are sorted from here on
    st->msd_ok = 1u;
    st->ss_ok = 1u;
  }
}

// Scatters each tile's keys (and labels) to their buckets: the tile's keys
// are staged in LDS in bucket order and each run is written by consecutive
// lanes at an atomic claim on the bucket's cursor.
template <typename K, bool LAB>
__global__ __launch_bounds__(kBlock) void ss_scatter_kernel(const K *__restrict__ in,
                                                            const uint32_t *__restrict__ vin,
                                                            K *__restrict__ out,
                                                            uint32_t *__restrict__ vout,
                                                            SsPlan p) {
  constexpr int IPT = Bk<K>::TIPT, TILE = kBlock * IPT;
  constexpr int PER = kSsMaxBuckets / kBlock;   // buckets per thread
  __shared__ K s_keys[TILE];
  __shared__ uint32_t s_vals[LAB ? TILE : 1];
  __shared__ uint16_t s_id[TILE];
  __shared__ uint32_t s_cnt[kSsMaxBuckets], s_lstart[kSsMaxBuckets], s_gstart[kSsMaxBuckets];
  __shared__ uint32_t s_w4[4];
  const uint32_t tile = blockIdx.x;
  if (p.limits && tile >= p.limits[0]) return;
  const uint32_t s = p.seg ? p.tiles.seg[tile] : 0u;
  const SsSeg sg = ss_segment(p, s);
  const uint32_t t = threadIdx.x;
  const uint32_t lo = (tile - (p.seg ? p.tiles.first[s] : 0u)) * (uint32_t)TILE;
  const uint32_t hi = min(lo + (uint32_t)TILE, sg.n);
#pragma unroll
  for (int i = 0; i < PER; ++i) s_cnt[t * PER + i] = 0;
  K k[IPT];
  uint32_t lv[IPT], dr[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = sg.kofs + (lo + j * kBlock + t < hi ? lo + j * kBlock + t : lo);
    k[j] = in[i];
    dr[j] = (uint32_t)p.ids[i] << 16;
    if (LAB) lv[j] = vin[i];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (lo + j * kBlock + t < hi) dr[j] |= atomicAdd(&s_cnt[dr[j] >> 16], 1u);
  __syncthreads();
  uint32_t c[PER], sum = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    c[i] = s_cnt[t * PER + i];
    sum += c[i];
  }
  uint32_t total;
  uint32_t ex = block_excl_sum<uint32_t>(sum, s_w4, &total);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const uint32_t b = t * PER + i;
    s_lstart[b] = ex;
    s_gstart[b] = c[i] ? atomicAdd(&p.cursors[sg.bucket + b], c[i]) : 0u;
    ex += c[i];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < IPT; ++j)
    if (lo + j * kBlock + t < hi) {
      const uint32_t b = dr[j] >> 16, q = s_lstart[b] + (dr[j] & 0xffffu);
      s_keys[q] = k[j];
      s_id[q] = (uint16_t)b;
      if (LAB) s_vals[q] = lv[j];
    }
  __syncthreads();
  const uint32_t end = sg.kofs + sg.n;
  for (uint32_t q = t; q < hi - lo; q += kBlock) {
    const uint32_t b = s_id[q];
    const uint32_t pos = s_gstart[b] + (q - s_lstart[b]);
    if (pos < end) {   // always true when the counts match the keys
      out[pos] = s_keys[q];
      if (LAB) vout[pos] = s_vals[q];
    }
  }
}

// Sorts each bucket (at most CAP keys) in LDS, from the buffer that holds it
// (kmid, or kin for a segment of one bucket; either may be kA) into kA (and
// vA) at its own positions, shifted by the segment's prepended
// key.  Reports equal neighbours, and a zero key at the front where one is
// prepended.
template <typename K, bool LAB, int BS, int IPT>
__global__ __launch_bounds__(BS) void ss_sort_kernel(const K *kin, const uint32_t *vin,
                                                     const K *kmid, const uint32_t *vmid, K *kA,
                                                     uint32_t *vA, SsPlan p, uint32_t prepend,
                                                     RunState *st) {
  constexpr int CAP = BS * IPT;
  __shared__ K s_keys[CAP];
  __shared__ uint32_t s_vals[LAB ? CAP : 1];
  __shared__ __align__(16) uint32_t s_tmp[bin_words<K, BS>()];
  if (p.limits && blockIdx.x >= p.limits[1]) return;
  const BkItem it = p.items[blockIdx.x];
  const uint32_t s0 = it.start, cnt = min(it.count, (uint32_t)CAP);
  if (cnt == 0) return;
  const K *in = it.parity ? kmid : kin;
  const uint32_t *lin = it.parity ? vmid : vin;
  const SsOut o = ss_out(p, it.sbits, prepend, st);
  const uint32_t t = threadIdx.x;
  K k[IPT];
  uint32_t v[IPT];
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = (uint32_t)j * BS + t;
    k[j] = i < cnt ? in[s0 + i] : kzero_value<K>();
    v[j] = (LAB && i < cnt) ? lin[s0 + i] : 0u;
  }
  lds_bin_sort<K, LAB, BS, IPT, (BS == 512 && sizeof(K) <= 8)>(
      k, v, cnt, [&](uint32_t i) { return in[s0 + i]; }, [&](uint32_t i) { return lin[s0 + i]; },
      s_keys, s_vals, s_tmp);
  __syncthreads();   // (every read of a bucket sorted in place is done too)
  bool dup = false;
#pragma unroll
  for (int j = 0; j < IPT; ++j) {
    const uint32_t i = (uint32_t)j * BS + t;
    if (i < cnt) {
      const K x = s_keys[i];
      dup |= i > 0 ? keq(x, s_keys[i - 1]) : (s0 == o.kofs && o.prepend && kzero(x));
      kA[s0 + o.shift + i] = x;
      if (LAB) vA[s0 + o.shift + i] = s_vals[i];
    }
  }
  if (__any(dup) && (t & 63) == 0) raise_flag(o.dups);
}

// Buckets above CAP, one workgroup to an item.  One key's copies are runs of up
// to CAP, each written from the first key of it (and its labels moved): many
// points at one place, as a scanner's missing returns leave them, spread over
// the chip like any others (one workgroup for all of them took a build of 2^24
// points, 5% of them at one place, from 875 to 1384 us).  Other buckets
// are a sample that misjudged them, a few in 10^6: stable LSD passes through
// global memory (the bucket's range of both buffers) over the bits that vary in
// it, slow beside the LDS sort.  Always reports duplicates: telling equal
// neighbours apart is left to unique.
template <typename K, bool LAB>
__global__ __launch_bounds__(kSsBlock) void ss_big_kernel(K *kmid, uint32_t *vmid, K *kA,
                                                          uint32_t *vA, K *kB, uint32_t *vB,
                                                          SsPlan p, RunState *st) {
  constexpr int NW = kSsBlock / 64;
  __shared__ uint32_t s_base[256], s_wc[NW * 256];
  __shared__ unsigned long long s_or[NW][4];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const uint32_t nbig = *p.n_big;
  for (uint32_t e = blockIdx.x; e < nbig; e += gridDim.x) {
    const BkItem it = p.big[e];
    const SsOut o = ss_out(p, it.sbits, 0u, st);
    if (t == 0) raise_flag(o.dups);
    if (it.parity == kSsBigRun) {   // uniform
      if (kmid == kA) continue;     // where they go already (no shift then)
      const K x = kmid[it.start];
      for (uint32_t i = t; i < it.count; i += kSsBlock) {
        kA[it.start + o.shift + i] = x;
        if (LAB) vA[it.start + o.shift + i] = vmid[it.start + i];
      }
      continue;
    }
    // from kmid (a big bucket was scattered: a segment of one bucket fits)
    // and the other buffer in turn, to end in A (shifted only where kmid is B)
    K *const outk = kA + o.shift;
    uint32_t *const outv = LAB ? vA + o.shift : nullptr;
    K *src = kmid, *dst = kmid == kA ? kB : outk;
    uint32_t *vsrc = vmid, *vdst = kmid == kA ? vB : outv;
    uint64_t olo = 0, ohi = 0, alo = ~0ull, ahi = ~0ull;
    for (uint32_t i = t; i < it.count; i += kSsBlock) {
      const K x = src[it.start + i];
      olo |= klo(x); ohi |= khi(x);
      alo &= klo(x); ahi &= khi(x);
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
      olo |= (uint64_t)__shfl_xor((unsigned long long)olo, d, 64);
      ohi |= (uint64_t)__shfl_xor((unsigned long long)ohi, d, 64);
      alo &= (uint64_t)__shfl_xor((unsigned long long)alo, d, 64);
      ahi &= (uint64_t)__shfl_xor((unsigned long long)ahi, d, 64);
    }
    __syncthreads();   // s_or and the counters are reused by every bucket
    if (lane == 0) { s_or[w][0] = olo; s_or[w][1] = ohi; s_or[w][2] = alo; s_or[w][3] = ahi; }
    __syncthreads();
    olo = 0; ohi = 0; alo = ~0ull; ahi = ~0ull;
    for (int ww = 0; ww < NW; ++ww) {
      olo |= s_or[ww][0]; ohi |= s_or[ww][1]; alo &= s_or[ww][2]; ahi &= s_or[ww][3];
    }
    const int passes = (varying_bits(olo, ohi, alo, ahi) + 7) / 8;   // uniform
    for (int q = 0; q < passes; ++q) {
      const int sh = 8 * q;
      if (t < 256) s_base[t] = 0;
      __syncthreads();
      for (uint32_t i = t; i < it.count; i += kSsBlock)
        atomicAdd(&s_base[kdigit(src[it.start + i], sh)], 1u);
      __syncthreads();
      if (t < 64) {   // exclusive scan of the 256 digit counts, four per lane
        uint32_t c[4], sum = 0;
        for (int j = 0; j < 4; ++j) { c[j] = s_base[4 * t + j]; sum += c[j]; }
        uint32_t run = wave_incl_scan_add(sum) - sum;
        for (int j = 0; j < 4; ++j) { s_base[4 * t + j] = run; run += c[j]; }
      }
      for (uint32_t base = 0; base < it.count; base += kSsBlock) {   // uniform
        for (int i = t; i < NW * 256; i += kSsBlock) s_wc[i] = 0;
        __syncthreads();
        const uint32_t i = base + t;
        const bool in = i < it.count;
        const K x = src[it.start + (in ? i : 0u)];
        const uint32_t d = kdigit(x, sh);
        uint64_t peers = __ballot(in);
        for (int b = 0; b < 8; ++b) {
          const uint64_t bb = __ballot((d >> b) & 1u);
          peers &= ((d >> b) & 1u) ? bb : ~bb;
        }
        const uint32_t below = (uint32_t)__popcll(peers & lanemask_lt());
        if (in && below == 0) s_wc[w * 256 + d] = (uint32_t)__popcll(peers);
        __syncthreads();
        if (t < 256) {   // the waves' starts within the digit, and the next tile's base
          uint32_t run = s_base[t];
          for (int ww = 0; ww < NW; ++ww) {
            const uint32_t c = s_wc[ww * 256 + t];
            s_wc[ww * 256 + t] = run;
            run += c;
          }
          s_base[t] = run;
        }
        __syncthreads();
        if (in) {
          const uint32_t pos = it.start + s_wc[w * 256 + d] + below;
          dst[pos] = x;
          if (LAB) vdst[pos] = vsrc[it.start + i];
        }
        __syncthreads();
      }
      __threadfence_block();
      __syncthreads();   // the pass is complete before the next reads it
      K *kt = src; src = dst; dst = kt;
      uint32_t *vt = vsrc; vsrc = vdst; vdst = vt;
    }
    if (src != outk) {
      for (uint32_t i = t; i < it.count; i += kSsBlock) {
        outk[it.start + i] = src[it.start + i];
        if (LAB) outv[it.start + i] = vsrc[it.start + i];
      }
    }
  }
}

__global__ __launch_bounds__(kBlock) void ss_zero_kernel(uint32_t *counts, uint32_t n,
                                                         uint32_t *n_big) {
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) counts[i] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) *n_big = 0;
}

}  // namespace

// Keys that a bucket averages: with 16 samples to a bucket and room for 2.5 times
// the average, one outgrows CAP where 40 expected samples drew 15 or fewer, some
// 5 buckets in 10^6.
template <typename K>
int64_t ss_bucket_keys() { return (int64_t)SsItem<K>::CAP * 40 / 100; }

template <typename K>
int64_t ss_max_keys() { return ss_bucket_keys<K>() * kSsMaxBuckets; }

template <typename K>
int ss_buckets(int64_t n) {
  if (n <= SsItem<K>::CAP) return 1;
  const int64_t T = ss_bucket_keys<K>();
  return n <= ss_max_keys<K>() ? (int)((n + T - 1) / T) : 0;
}

template <typename K>
int ss_tile() { return kBlock * Bk<K>::TIPT; }

template <typename K>
size_t ss_ws_bytes(int64_t buckets, int64_t segs, int64_t slots) {
  return align256_dev((size_t)buckets * sizeof(K)) +
         align256_dev((size_t)segs * kSsLutWords * 4) +
         2 * align256_dev((size_t)buckets * 4) + align256_dev((size_t)buckets * sizeof(BkItem)) +
         align256_dev((size_t)buckets * 2 * sizeof(BkItem)) +
         align256_dev((size_t)slots * 2) + 256;
}

template <typename K>
void ss_carve(void *ws, int64_t buckets, int64_t segs, int64_t slots, SsPlan &p) {
  char *q = static_cast<char *>(ws);
  auto take = [&](size_t bytes) { char *r = q; q += align256_dev(bytes); return r; };
  p.splitters = take((size_t)buckets * sizeof(K));
  p.lut = reinterpret_cast<uint32_t *>(take((size_t)segs * kSsLutWords * 4));
  p.counts = reinterpret_cast<uint32_t *>(take((size_t)buckets * 4));
  p.cursors = reinterpret_cast<uint32_t *>(take((size_t)buckets * 4));
  p.items = reinterpret_cast<BkItem *>(take((size_t)buckets * sizeof(BkItem)));
  // (a bucket of c keys gives at most max(1, 2 c / CAP) items, and a bucket
  // averages 0.4 CAP keys)
  p.big = reinterpret_cast<BkItem *>(take((size_t)buckets * 2 * sizeof(BkItem)));
  p.ids = reinterpret_cast<uint16_t *>(take((size_t)slots * 2));
  p.n_big = reinterpret_cast<uint32_t *>(take(4));
  p.n_buckets = buckets;
  p.n_segs = segs;
}

// The crowded buckets' tables, at most S segments: SegInfo[S], first tiles
// and first buckets (S + 1 each), the two limits, tile -> segment.
struct SsTables {
  SegInfo *seg;
  uint32_t *tile_first, *bucket_first, *limits, *tile_seg;
};
inline SsTables ss_tables(void *ws, int64_t S) {
  char *q = static_cast<char *>(ws);
  auto take = [&](size_t bytes) { char *r = q; q += align256_dev(bytes); return r; };
  SsTables t;
  t.seg = reinterpret_cast<SegInfo *>(take((size_t)S * sizeof(SegInfo)));
  t.tile_first = reinterpret_cast<uint32_t *>(take((size_t)(S + 1) * 4));
  t.bucket_first = reinterpret_cast<uint32_t *>(take((size_t)(S + 1) * 4));
  t.limits = reinterpret_cast<uint32_t *>(take(8));
  t.tile_seg = reinterpret_cast<uint32_t *>(q);
  return t;
}
// (a crowded bucket holds more than the bucket sort's CAP keys)
template <typename K>
int64_t ss_crowded_segs(int64_t n) { return n / Bk<K>::CAP + 2; }
template <typename K>
int64_t ss_crowded_buckets(int64_t n) { return n / ss_bucket_keys<K>() + ss_crowded_segs<K>(n); }
template <typename K>
int64_t ss_crowded_tiles(int64_t n) { return n / ss_tile<K>() + ss_crowded_segs<K>(n); }

template <typename K>
size_t ss_tree_bytes(int64_t n) {
  const int64_t S = ss_crowded_segs<K>(n);
  const size_t tables = align256_dev((size_t)S * sizeof(SegInfo)) +
                        2 * align256_dev((size_t)(S + 1) * 4) + align256_dev(8) +
                        align256_dev((size_t)ss_crowded_tiles<K>(n) * 4);
  return tables + ss_ws_bytes<K>(ss_crowded_buckets<K>(n), S, n);
}

template <typename K>
void ss_tree_carve(void *ws, int64_t n, SsTree &t) {
  const int64_t S = ss_crowded_segs<K>(n);
  const size_t tables = ss_tree_bytes<K>(n) - ss_ws_bytes<K>(ss_crowded_buckets<K>(n), S, n);
  char *rest = static_cast<char *>(ws) + tables;
  t.tables = ws;
  ss_carve<K>(rest, ss_crowded_buckets<K>(n), S, n, t.crowded);
  const int nb = ss_buckets<K>(n);
  if (nb > 1) {
    ss_carve<K>(rest, nb, 1, n, t.whole);
    t.whole.n = (uint32_t)n;
    t.whole.nb = t.whole.max_nb = (uint32_t)nb;
    t.whole.n_tiles = (n + ss_tile<K>() - 1) / ss_tile<K>();
  }
}

// One workgroup: the tables of the nseg crowded buckets segs[].  mostly: where
// they hold more than a quarter of the n keys, the sample sort, not the bucket
// sort, is reported to have sorted them.
__global__ __launch_bounds__(kSsBlock) void ss_tables_kernel(const BkSeg *__restrict__ segs,
                                                             uint32_t nseg, uint32_t T,
                                                             uint32_t tile, uint32_t n,
                                                             int mostly, SsTables o,
                                                             RunState *st) {
  __shared__ uint32_t s_w[kSsBlock / 64];
  uint32_t tiles = 0, buckets = 0;   // before this round's segments (uniform)
  for (uint32_t base = 0; base < nseg; base += kSsBlock) {
    const uint32_t i = base + threadIdx.x;
    const uint32_t cnt = i < nseg ? segs[i].count : 0u;
    const uint32_t nt = (cnt + tile - 1) / tile, nb = (cnt + T - 1) / T;
    uint32_t all_t, all_b;
    const uint32_t ft = tiles + block_excl_sum<uint32_t, kSsBlock / 64>(nt, s_w, &all_t);
    __syncthreads();   // s_w is reused
    const uint32_t fb = buckets + block_excl_sum<uint32_t, kSsBlock / 64>(nb, s_w, &all_b);
    __syncthreads();
    if (i < nseg) {
      SegInfo x{};
      x.n = cnt;
      x.kofs = segs[i].start;
      o.seg[i] = x;
      o.tile_first[i] = ft;
      o.bucket_first[i] = fb;
      for (uint32_t k = 0; k < nt; ++k) o.tile_seg[ft + k] = i;
    }
    tiles += all_t;
    buckets += all_b;
  }
  if (threadIdx.x == 0) {
    o.tile_first[nseg] = tiles;
    o.bucket_first[nseg] = buckets;
    o.limits[0] = tiles;
    o.limits[1] = buckets;
    st->msd_ok = 1u;   // (sorted from here on)
    if (mostly && (uint64_t)st->bk_keys * 4 > n) st->ss_ok = 1u;
  }
}

template <typename K, int CAP, int BS>
void ss_sort(const K *kin, const uint32_t *vin, const K *kmid, const uint32_t *vmid, K *kA,
             uint32_t *vA, const SsPlan &p, int prepend, RunState *st, hipStream_t s) {
  const unsigned items = (unsigned)p.n_buckets;
  if (vin)
    ss_sort_kernel<K, true, BS, CAP / BS><<<items, BS, 0, s>>>(kin, vin, kmid, vmid, kA, vA, p,
                                                               (uint32_t)prepend, st);
  else
    ss_sort_kernel<K, false, BS, CAP / BS><<<items, BS, 0, s>>>(kin, nullptr, kmid, nullptr, kA,
                                                                nullptr, p, (uint32_t)prepend, st);
}

template <typename K>
void launch_sample_sort(const K *kin, const uint32_t *vin, K *kA, uint32_t *vA, K *kB,
                        uint32_t *vB, const SsPlan &p, int mbits, int prepend, RunState *st,
                        hipStream_t s) {
  K *kmid = kin == kA ? kB : kA;
  uint32_t *vmid = kin == kA ? vB : vA;
  const unsigned segs = (unsigned)p.n_segs, tiles = (unsigned)p.n_tiles;
  const unsigned zgrid = (unsigned)std::min<int64_t>((p.n_buckets + kBlock - 1) / kBlock, 1024);
  if (segs) {
    ss_zero_kernel<<<zgrid, kBlock, 0, s>>>(p.counts, (uint32_t)p.n_buckets, p.n_big);
    if (p.max_nb <= kSsMaxBuckets / 4)
      ss_splitters_kernel<K, kSsIpt / 4><<<segs, kSsBlock, 0, s>>>(kin, p, mbits);
    else if (p.max_nb <= kSsMaxBuckets / 2)
      ss_splitters_kernel<K, kSsIpt / 2><<<segs, kSsBlock, 0, s>>>(kin, p, mbits);
    else
      ss_splitters_kernel<K, kSsIpt><<<segs, kSsBlock, 0, s>>>(kin, p, mbits);
    ss_count_kernel<K><<<tiles, kBlock, 0, s>>>(kin, p, mbits);
    const uint32_t cap = (uint32_t)SsItem<K>::CAP;
    ss_plan_kernel<K><<<segs, kSsMaxBuckets, 0, s>>>(
        p, p.item_keys ? std::min(p.item_keys, cap) : cap, mbits, st);
    if (vin)
      ss_scatter_kernel<K, true><<<tiles, kBlock, 0, s>>>(kin, vin, kmid, vmid, p);
    else
      ss_scatter_kernel<K, false><<<tiles, kBlock, 0, s>>>(kin, nullptr, kmid, nullptr, p);
  }
  // Few buckets leave the chip to one workgroup per CU or less: then twice
  // the threads on each (300,000 keys: 170 against 181 us a build); with many,
  // two workgroups of half of them on each CU (55 M keys: 3.03 against 3.35 ms
  // a batch).
  constexpr int CAP = SsItem<K>::CAP;
  if (p.n_buckets <= 512)
    ss_sort<K, CAP, 1024>(kin, vin, kmid, vmid, kA, vA, p, prepend, st, s);
  else
    ss_sort<K, CAP, 512>(kin, vin, kmid, vmid, kA, vA, p, prepend, st, s);
  if (!segs) return;
  if (vin)
    ss_big_kernel<K, true><<<kSsBigGrid, kSsBlock, 0, s>>>(kmid, vmid, kA, vA, kB, vB, p, st);
  else
    ss_big_kernel<K, false><<<kSsBigGrid, kSsBlock, 0, s>>>(kmid, nullptr, kA, nullptr, kB, nullptr, p, st);
}

template <typename K>
void launch_sample_sort_buckets(const K *kin, const uint32_t *vin, K *kA, uint32_t *vA, K *kB,
                                uint32_t *vB, const SsTree &t, const BkSeg *segs, uint32_t nseg,
                                uint64_t nkeys, uint32_t max_keys, int64_t n, int mbits,
                                int prepend, uint32_t item_keys, RunState *st, hipStream_t s) {
  const SsTables o = ss_tables(t.tables, ss_crowded_segs<K>(n));
  const uint32_t T = (uint32_t)ss_bucket_keys<K>();
  ss_tables_kernel<<<1, kSsBlock, 0, s>>>(segs, nseg, T, (uint32_t)ss_tile<K>(), (uint32_t)n,
                                          sizeof(K) <= 8 ? 1 : 0, o, st);
  SsPlan p = t.crowded;
  p.item_keys = item_keys;
  p.seg = o.seg;
  p.tiles.seg = o.tile_seg;
  p.tiles.first = o.tile_first;
  p.bucket_first = o.bucket_first;
  p.limits = o.limits;
  p.n_segs = nseg;
  p.n_tiles = (int64_t)(nkeys / ss_tile<K>()) + nseg;
  p.n_buckets = (int64_t)(nkeys / T) + nseg;
  p.max_nb = (max_keys + T - 1) / T;
  launch_sample_sort<K>(kin, vin, kA, vA, kB, vB, p, mbits, prepend, st, s);
}

#define PGVD_SS_INST(K)                                                                       \
  template int ss_buckets<K>(int64_t);                                                        \
  template int64_t ss_max_keys<K>();                                                          \
  template int ss_tile<K>();                                                                  \
  template size_t ss_ws_bytes<K>(int64_t, int64_t, int64_t);                                  \
  template void ss_carve<K>(void *, int64_t, int64_t, int64_t, SsPlan &);                     \
  template size_t ss_tree_bytes<K>(int64_t);                                                  \
  template void ss_tree_carve<K>(void *, int64_t, SsTree &);                                  \
  template void launch_sample_sort<K>(const K *, const uint32_t *, K *, uint32_t *, K *,      \
                                      uint32_t *, const SsPlan &, int, int, RunState *,       \
                                      hipStream_t);                                           \
  template void launch_sample_sort_buckets<K>(const K *, const uint32_t *, K *, uint32_t *,   \
                                              K *, uint32_t *, const SsTree &, const BkSeg *, \
                                              uint32_t, uint64_t, uint32_t, int64_t, int,     \
                                              int, uint32_t, RunState *, hipStream_t);
PGVD_SS_INST(uint32_t)
PGVD_SS_INST(uint64_t)
PGVD_SS_INST(Key128)
#undef PGVD_SS_INST

}  // namespace pgvd
