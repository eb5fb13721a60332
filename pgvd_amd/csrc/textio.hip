// textio.hip -- the octree's text form on the device: operator<< and
// operator>> for OctNode and std::vector<OctNode> (C/OctNode.h:58-98,
// commented out in the reference).  The text is "N " followed, for every
// node, by each child and the leaf mask in decimal, each followed by one
// space.
//
// Both directions are one pass with a decoupled look-back over tiles:
//   format: a workgroup takes 4 x 256 nodes, sums their text lengths, scans
//           them in the workgroup and across tiles, and prints each 256 into
//           LDS and copies the run out at its offset in turn;
//   parse:  a workgroup takes 4 x 8192 bytes, marks where tokens start
//           (a non-space after a space), scans the counts to token numbers,
//           lists the starts, and parses the tokens from LDS one to a lane,
//           token k into value k - 1 (token 0 is N, read by the host).
#include "kernels.hpp"
#include "tilescan.hpp"

namespace pgvd {

namespace {

// workspace words (uint64): [0] tile counter (low 32 bits), [1] total
// (bytes or tokens, written by the last tile), [2] first malformed token + 1
// (atomic min over ~0: none), then the tile status array from word 4.
constexpr int kWsCounter = 0, kWsTotal = 1, kWsBad = 2, kWsStatus = 4;
constexpr int kFmtBlock = 256;        // nodes per format tile
constexpr int kMaxNodeText = 9 * 12;  // 3D node: 9 values of at most 11 chars + space
constexpr int kParseBytes = 16;       // bytes per thread in a parse tile
#ifndef PGVD_PARSE_BLOCK
#define PGVD_PARSE_BLOCK 512
#endif
constexpr int kParseBlock = PGVD_PARSE_BLOCK;   // threads per parse workgroup
constexpr int kParseTile = kParseBlock * kParseBytes;   // bytes per round
#ifndef PGVD_PARSE_ROUNDS
#define PGVD_PARSE_ROUNDS 4
#endif
constexpr int kParseRounds = PGVD_PARSE_ROUNDS;          // rounds per tile
static_assert(kParseRounds >= 1 && kParseRounds <= 4, "start counts are packed in 16-bit fields");

__device__ inline int dec_len(int32_t v) {
  uint32_t u = v < 0 ? 0u - (uint32_t)v : (uint32_t)v;
  int n = 1;
  if (u >= 10u) n = 2;
  if (u >= 100u) n = 3;
  if (u >= 1000u) n = 4;
  if (u >= 10000u) n = 5;
  if (u >= 100000u) n = 6;
  if (u >= 1000000u) n = 7;
  if (u >= 10000000u) n = 8;
  if (u >= 100000000u) n = 9;
  if (u >= 1000000000u) n = 10;
  return n + (v < 0);
}

// Prints v, n = dec_len(v) characters, and one space at s[at..]; returns the
// position after the space.  Two digits a step: their values come from one
// multiplication and a table of the 100 pairs.
__device__ inline int put_dec(uint8_t *s, int at, int32_t v, int n, const uint16_t *pairs) {
  uint32_t u = v < 0 ? 0u - (uint32_t)v : (uint32_t)v;
  int e = at + n;
  s[e] = ' ';
  while (u >= 10u) {
    const uint32_t q = u / 100u, two = pairs[u - q * 100u];
    s[--e] = (uint8_t)(two >> 8);
    s[--e] = (uint8_t)two;
    u = q;
  }
  // a digit is left, or none (an even number of them is out, unless v is 0)
  if (e > at + (v < 0)) s[--e] = (uint8_t)('0' + u);
  if (v < 0) s[at] = '-';
  return at + n + 1;
}

__global__ void ws_zero_kernel(uint64_t *ws, int64_t words) {
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < words;
       i += (int64_t)gridDim.x * kBlock)
    ws[i] = i == kWsBad ? ~0ull : 0ull;
}

#ifndef PGVD_FMT_ROUNDS
#define PGVD_FMT_ROUNDS 4
#endif
constexpr int kFmtRounds = PGVD_FMT_ROUNDS;   // 256-node rounds per tile
static_assert(kFmtRounds >= 1 && kFmtRounds <= 4, "round lengths are packed in 16-bit fields");

// A tile is kFmtRounds rounds of 256 nodes with one look-back: the rounds'
// text lengths are scanned together as 16-bit fields of one word (a round
// holds at most 256 * 108 bytes, below 2^16), then each round is printed
// into LDS, from the byte that its run begins at in a 16-byte line of the
// text, and the lines are copied out whole (the first and last by bytes).
// What bounds it is the byte stores into LDS and the digits' arithmetic; an
// octree of 2^22 uniform 3D points takes 91 us (106 with a division for each
// digit, the lengths found twice and words put together from bytes).
template <int DIM>
__global__ __launch_bounds__(kFmtBlock) void format_text_kernel(
    const int32_t *__restrict__ octree, int64_t O, int64_t N_hdr, int hdr_len,
    uint8_t *__restrict__ text, int64_t capacity, uint64_t *__restrict__ ws, int ntiles) {
  constexpr int STRIDE = (1 << DIM) + 1;
  __shared__ __align__(16) uint8_t s_txt[kFmtBlock * kMaxNodeText + 16];
  __shared__ uint16_t s_pairs[100];
  __shared__ uint64_t s_w[kFmtBlock / 64];
  __shared__ int s_tile;
  const int t = threadIdx.x;
  if (t == 0) s_tile = (int)atomicAdd(reinterpret_cast<unsigned int *>(ws + kWsCounter), 1u);
  if (t < 100) s_pairs[t] = (uint16_t)((uint32_t)('0' + t / 10) | (uint32_t)('0' + t % 10) << 8);
  __syncthreads();
  const int tile = s_tile;
  const int64_t first = (int64_t)tile * kFmtBlock * kFmtRounds;
  uint64_t packed = 0;
  uint64_t lens[kFmtRounds];   // the values' lengths, 4 bits each
  int32_t cur[STRIDE];   // the records of the round being printed (round 0 kept from here)
#pragma unroll
  for (int r = 0; r < kFmtRounds; ++r) {
    const int64_t i = first + r * kFmtBlock + t;
    uint32_t len = 0;
    lens[r] = 0;
#pragma unroll
    for (int k = 0; k < STRIDE; ++k) {
      const int32_t x = i < O ? octree[i * STRIDE + k] : 0;
      if (r == 0) cur[k] = x;
      const int n = dec_len(x);
      lens[r] |= (uint64_t)n << (4 * k);
      len += (uint32_t)n + 1u;
    }
    packed |= (uint64_t)(i < O ? len : 0u) << (16 * r);
  }
  uint64_t tot_packed;
  const uint64_t ex = block_excl_sum<uint64_t, kFmtBlock / 64>(packed, s_w, &tot_packed);
  uint32_t total = 0;
#pragma unroll
  for (int r = 0; r < kFmtRounds; ++r) total += (uint32_t)(tot_packed >> (16 * r)) & 0xffffu;
  const uint64_t before = tile_prefix<kFmtBlock>(ws + kWsStatus, tile, total);
  if (tile == ntiles - 1 && t == 0) ws[kWsTotal] = (uint64_t)hdr_len + before + total;
  if (!text) return;
  int64_t g0 = hdr_len + (int64_t)before;
  if (g0 + (int64_t)total > capacity) return;
  if (tile == 0 && t == 0) {
    // "N " at the start: N printed from the least significant digit
    uint64_t u = (uint64_t)N_hdr;
    int e = hdr_len - 1;
    text[e] = ' ';
    do {
      text[--e] = (uint8_t)('0' + u % 10u);
      u /= 10u;
    } while (u);
  }
#pragma unroll
  for (int r = 0; r < kFmtRounds; ++r) {
    const int rtotal = (int)((uint32_t)(tot_packed >> (16 * r)) & 0xffffu);
    const int64_t i = first + r * kFmtBlock + t;
    // the next round's records load while this round prints
    int32_t nxt[STRIDE];
    const int64_t in = i + kFmtBlock;
#pragma unroll
    for (int k = 0; k < STRIDE; ++k)
      nxt[k] = (r + 1 < kFmtRounds && in < O) ? octree[in * STRIDE + k] : 0;
    const int lead = (int)((uintptr_t)(text + g0) & 15);
    if (r > 0) __syncthreads();   // the previous round's copy has read s_txt
    if (i < O) {
      int at = lead + (int)((ex >> (16 * r)) & 0xffffu);
#pragma unroll
      for (int k = 0; k < STRIDE; ++k)
        at = put_dec(s_txt, at, cur[k], (int)(lens[r] >> (4 * k)) & 15, s_pairs);
    }
    __syncthreads();
    // s_txt[lead, end) is the run; line w is its bytes 16 w .. 16 w + 15
    uint8_t *dst = text + g0 - lead;
    const int end = lead + rtotal;
    const int w0 = lead ? 1 : 0, w1 = end >> 4;
    for (int w = w0 + t; w < w1; w += kFmtBlock)
      reinterpret_cast<uint4 *>(dst)[w] = reinterpret_cast<const uint4 *>(s_txt)[w];
    if (t < 16) {
      if (lead && t >= lead && t < end) dst[t] = s_txt[t];
      const int b = 16 * w1 + t;
      if (w1 >= w0 && b < end) dst[b] = s_txt[b];
    }
    g0 += rtotal;
#pragma unroll
    for (int k = 0; k < STRIDE; ++k) cur[k] = nxt[k];
  }
}

// ' ', '\t', '\n', '\v', '\f', '\r' (codes 32 and 9..13) as one mask test
__device__ inline bool is_space(uint8_t c) {
  return c <= 32 && ((0x100003E00ull >> c) & 1ull);
}

// Bits 0..3: which of w's four bytes are spaces.
__device__ inline uint32_t space_bits(uint32_t w) {
  const uint32_t lo = w & 0x7f7f7f7fu;                       // no sum below carries
  const uint32_t from9 = lo + 0x77777777u, from14 = lo + 0x72727272u;
  const uint32_t not32 = (lo ^ 0x20202020u) + 0x7f7f7f7fu;
  const uint32_t m = ((from9 & ~from14) | ~not32) & ~w & 0x80808080u;
  return ((m >> 7) * 0x01020408u) >> 24;                     // bits 0, 8, 16, 24 -> 24..27
}

// Four decimal digits, the first in the lowest byte.
__device__ inline uint32_t digits4(uint32_t d) {
  return __builtin_amdgcn_udot4(d, 0x010Au, 0u, false) * 100u +
         __builtin_amdgcn_udot4(d, 0x010A0000u, 0u, false);
}

// The common token at byte p of s, which has 12 bytes after p: an optional
// minus, 1 to 8 digits and a space.  The digits are found and added up four
// to a word; false where the token has another form (parse_staged decides).
__device__ inline bool parse_short(const uint8_t *s, int p, int32_t *out) {
  const uint32_t *q = reinterpret_cast<const uint32_t *>(s) + (p >> 2);
  const uint32_t q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3], sh = (uint32_t)p & 3u;
  uint32_t w0 = __builtin_amdgcn_alignbyte(q1, q0, sh), w1 = __builtin_amdgcn_alignbyte(q2, q1, sh),
           w2 = __builtin_amdgcn_alignbyte(q3, q2, sh);
  const uint32_t neg = (w0 & 0xffu) == '-' ? 1u : 0u;
  w0 = __builtin_amdgcn_alignbyte(w1, w0, neg);
  w1 = __builtin_amdgcn_alignbyte(w2, w1, neg);
  w2 = __builtin_amdgcn_alignbyte(0u, w2, neg);
  // bit 7 of each byte: no digit (right up to the first such byte)
  const uint32_t x0 = w0 ^ 0x30303030u, x1 = w1 ^ 0x30303030u;
  const uint32_t m0 = ((x0 + 0x76767676u) | x0) & 0x80808080u;
  const uint32_t m1 = ((x1 + 0x76767676u) | x1) & 0x80808080u;
  const uint32_t n = m0 ? (uint32_t)__builtin_ctz(m0) >> 3
                        : (m1 ? 4u + ((uint32_t)__builtin_ctz(m1) >> 3) : 8u);
  const uint32_t endw = n < 4 ? w0 : (n < 8 ? w1 : w2);
  if (n == 0 || !is_space((uint8_t)(endw >> (8 * (n & 3u))))) return false;
  const uint64_t d = ((uint64_t)x1 << 32 | x0) << (8 * (8 - n));   // right-aligned, zeros before
  const uint32_t v = digits4((uint32_t)d) * 10000u + digits4((uint32_t)(d >> 32));
  *out = neg ? -(int32_t)v : (int32_t)v;
  return true;
}

// Token parse from the staged bytes: an optional sign and digits, at most
// 10 of them significant (leading zeros are skipped, as operator>> skips
// them), ending at a space (bytes past the text read as spaces), within
// int32.  A token running past the staged bytes (only one with leading
// zeros can) continues from global memory: byte q of s is text[g0 + q].
__device__ inline bool parse_staged(const uint8_t *s, int p, int staged, const uint8_t *text,
                                    int64_t g0, int64_t len, int32_t *out) {
  auto at = [&](int q) -> uint8_t {
    if (q < staged) return s[q];
    return g0 + q < len ? text[g0 + q] : (uint8_t)' ';
  };
  bool neg = false;
  uint8_t c = at(p);
  if (c == '+' || c == '-') {
    neg = c == '-';
    ++p;
  }
  int64_t x = 0;
  int nd = 0;
  bool digit = false;
  for (;; ++p) {
    c = at(p);
    if (is_space(c)) break;
    if (c < '0' || c > '9') return false;
    digit = true;
    if (nd == 0 && c == '0') continue;
    if (nd >= 10) return false;
    x = x * 10 + (c - '0');
    ++nd;
  }
  if (!digit) return false;
  if (neg) x = -x;
  if (x < INT32_MIN || x > INT32_MAX) return false;
  *out = (int32_t)x;
  return true;
}

// A tile is kParseRounds rounds of kParseTile bytes with one look-back: the
// rounds' token-start counts are scanned together as 16-bit fields of one
// word (a round holds at most kParseTile / 2 starts), then each round's
// bytes and the 16 after it are staged in LDS (a token starting in the round
// without leading zeros is decided within 12 bytes: sign, 10 digits, one
// more byte; a longer one reads on from global memory), the starts listed in
// token order, and the tokens parsed one to a lane, each lane writing its
// value where it belongs, next to its neighbours'.  What bounds it is the
// VALU: tokens differ in number per 16 bytes and in length, so neither the
// bytes' owners (which held a wave for its most crowded 16 bytes) nor a loop
// over digits divides them evenly.  The text of an octree of 2^22 uniform 3D
// points: 259 us by owners and digit by digit, 79 us so.
template <int DIM>
__global__ __launch_bounds__(kParseBlock) void parse_text_kernel(
    const uint8_t *__restrict__ text, int64_t len, int64_t N, int32_t *__restrict__ octree,
    uint64_t *__restrict__ ws, int ntiles) {
  constexpr uint32_t STRIDE = (1 << DIM) + 1;
  constexpr int kHalo = 16;
  __shared__ __align__(16) uint8_t s_txt[kParseTile + kHalo];
  __shared__ uint16_t s_pos[kParseTile / 2];
  __shared__ uint64_t s_w[kParseBlock / 64];
  __shared__ int s_tile;
  const int t = threadIdx.x;
  if (t == 0) s_tile = (int)atomicAdd(reinterpret_cast<unsigned int *>(ws + kWsCounter), 1u);
  __syncthreads();
  const int tile = s_tile;
  const int64_t tb = (int64_t)tile * kParseTile * kParseRounds;
  uint4 qs[kParseRounds];          // this thread's bytes of every round
  uint32_t smask[kParseRounds];    // and where tokens start in them
#pragma unroll
  for (int r = 0; r < kParseRounds; ++r) {
    const int64_t p0 = tb + (int64_t)r * kParseTile + (int64_t)t * kParseBytes;
    if (p0 + kParseBytes <= len && (((uintptr_t)(text + p0)) & 15) == 0) {
      qs[r] = *reinterpret_cast<const uint4 *>(text + p0);
    } else {
      uint32_t wv[4] = {0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < kParseBytes; ++k)
        wv[k >> 2] |= (uint32_t)(p0 + k < len ? text[p0 + k] : (uint8_t)' ') << (8 * (k & 3));
      qs[r] = make_uint4(wv[0], wv[1], wv[2], wv[3]);
    }
  }
  // threads below kHalo: byte t after the tile
  const int64_t ph = tb + (int64_t)kParseRounds * kParseTile + t;
  const uint8_t halo = (t < kHalo && ph < len) ? text[ph] : (uint8_t)' ';
  uint64_t packed = 0;
#pragma unroll
  for (int r = 0; r < kParseRounds; ++r) {
    const int64_t p0 = tb + (int64_t)r * kParseTile + (int64_t)t * kParseBytes;
    const uint32_t sp = space_bits(qs[r].x) | space_bits(qs[r].y) << 4 |
                        space_bits(qs[r].z) << 8 | space_bits(qs[r].w) << 12;
    uint32_t prev = __shfl_up(sp >> 15, 1, 64);   // is the byte before this thread's a space?
    if ((t & 63) == 0) prev = p0 == 0 || p0 > len || is_space(text[p0 - 1]);
    smask[r] = ~sp & (sp << 1 | prev) & 0xffffu;
    packed |= (uint64_t)__popc(smask[r]) << (16 * r);
  }
  uint64_t tot_packed;
  const uint64_t ex = block_excl_sum<uint64_t, kParseBlock / 64>(packed, s_w, &tot_packed);
  uint32_t total = 0;
#pragma unroll
  for (int r = 0; r < kParseRounds; ++r) total += (uint32_t)(tot_packed >> (16 * r)) & 0xffffu;
  const uint64_t before = tile_prefix<kParseBlock>(ws + kWsStatus, tile, total);
  if (tile == ntiles - 1 && t == 0) ws[kWsTotal] = before + total;
  const uint64_t last = (uint64_t)N * STRIDE;   // tokens 1..last are the records
  uint64_t base = before;
#pragma unroll
  for (int r = 0; r < kParseRounds; ++r) {
    const uint32_t rtotal = (uint32_t)(tot_packed >> (16 * r)) & 0xffffu;
    if (r > 0) __syncthreads();   // the previous round is done with s_txt and s_pos
    *reinterpret_cast<uint4 *>(s_txt + t * kParseBytes) = qs[r];
    if (r + 1 < kParseRounds) {
      if (t == 0) *reinterpret_cast<uint4 *>(s_txt + kParseTile) = qs[r + 1 < kParseRounds ? r + 1 : r];
    } else if (t < kHalo) {
      s_txt[kParseTile + t] = halo;
    }
    uint32_t li = (uint32_t)(ex >> (16 * r)) & 0xffffu;
    for (uint32_t starts = smask[r]; starts; starts &= starts - 1)
      s_pos[li++] = (uint16_t)(t * kParseBytes + __ffs(starts) - 1);
    __syncthreads();
    // token base + i is value k - 1 of the records: its column by 32-bit steps
    const uint32_t col0 = (uint32_t)((base + STRIDE - 1) % STRIDE);
    for (uint32_t i = t; i < rtotal; i += kParseBlock) {
      const uint64_t k = base + i;
      if (k < 1 || k > last) continue;
      int32_t v = 0;
      const int p = s_pos[i];
      if (!parse_short(s_txt, p, &v) &&
          !parse_staged(s_txt, p, kParseTile + kHalo, text, tb + (int64_t)r * kParseTile, len, &v)) {
        v = 0;
        atomicMin(reinterpret_cast<unsigned long long *>(ws + kWsBad), (unsigned long long)k + 1);
      }
      octree[k - 1] = (col0 + i) % STRIDE == STRIDE - 1 ? (int32_t)(uint8_t)v : v;
    }
    base += rtotal;
  }
}

}  // namespace

int64_t text_ws_words(int64_t tiles) { return kWsStatus + tiles; }
int64_t format_text_tiles(int64_t O) {
  return (O + kFmtBlock * kFmtRounds - 1) / (kFmtBlock * kFmtRounds);
}
int64_t parse_text_tiles(int64_t len) {
  return (len + (int64_t)kParseTile * kParseRounds - 1) / ((int64_t)kParseTile * kParseRounds);
}

void launch_format_text(const int32_t *octree, int64_t O, int dim, int hdr_len, uint8_t *text,
                        int64_t capacity, uint64_t *ws, hipStream_t s) {
  const int64_t tiles = format_text_tiles(O);
  const int64_t words = text_ws_words(tiles);
  ws_zero_kernel<<<(unsigned)std::min<int64_t>((words + kBlock - 1) / kBlock, 1024), kBlock, 0,
                   s>>>(ws, words);
  if (dim == 2)
    format_text_kernel<2><<<(unsigned)tiles, kFmtBlock, 0, s>>>(octree, O, O, hdr_len, text,
                                                                capacity, ws, (int)tiles);
  else
    format_text_kernel<3><<<(unsigned)tiles, kFmtBlock, 0, s>>>(octree, O, O, hdr_len, text,
                                                                capacity, ws, (int)tiles);
}

void launch_parse_text(const uint8_t *text, int64_t len, int dim, int64_t N, int32_t *octree,
                       uint64_t *ws, hipStream_t s) {
  const int64_t tiles = parse_text_tiles(len);
  const int64_t words = text_ws_words(tiles);
  ws_zero_kernel<<<(unsigned)std::min<int64_t>((words + kBlock - 1) / kBlock, 1024), kBlock, 0,
                   s>>>(ws, words);
  if (dim == 2)
    parse_text_kernel<2><<<(unsigned)tiles, kParseBlock, 0, s>>>(text, len, N, octree, ws,
                                                                 (int)tiles);
  else
    parse_text_kernel<3><<<(unsigned)tiles, kParseBlock, 0, s>>>(text, len, N, octree, ws,
                                                                 (int)tiles);
}

}  // namespace pgvd
