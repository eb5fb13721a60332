// walk.hip -- batched cell walks: CellWalk (viewer/Octree2.cpp:265-313) for
// many 2D segments at once, one lane per segment.  Each step locates the
// current point's leaf (FindLeaf with the octant masked to two bits), visits
// it, intersects the segment with the cell's four edges
// (OctreeUtils::FindIntersections, OctreeUtils.cpp:80-172) and moves to the
// farthest intersection.
//
// The walk's length is not known in advance, so a batch runs it twice: a
// counting pass, a scan of the counts to offsets (decoupled look-back), and
// a pass that writes every visited cell at its segment's offset.  The float
// arithmetic follows the reference operation by operation (no contraction,
// correctly rounded division and square root, epsilon tests in double), so
// both passes and the serial restatement visit the same cells.
#include "kernels.hpp"
#include "tilescan.hpp"
#include "walk_geom.hpp"

namespace pgvd {

namespace {

constexpr int kWalkMax = 10000;        // the reference throws past this many cells

// FindLeaf of the truncated point (convert_int2); cell = origin x, origin
// y, width, parent, octant.
__device__ inline void walk_leaf(float px, float py, int bits, const int32_t *__restrict__ octree,
                                 int64_t size, int32_t cell[5]) {
  const int32_t qx = (int32_t)px, qy = (int32_t)py;
  const int64_t c[2] = {qx, qy};
  uint64_t lo, hi;
  morton128<2>(c, bits, lo, hi);
  int64_t idx = 0;
  uint32_t o = 0;
  int32_t lev = 0;
  for (int sh = 2 * bits - 2; sh >= 0; sh -= 2) {
    o = (uint32_t)(lo >> sh) & 3u;
    ++lev;
    const int32_t *node = octree + idx * 5;
    const int32_t child = node[o];
    if ((node[4] >> o) & 1) break;
    if (child < 0 || child >= size) break;
    idx = child;
  }
  const int32_t w = (int32_t)(1u << (bits - lev));
  const int32_t gmask = (int32_t)((1u << bits) - 1);
  cell[0] = (qx & gmask) & ~(w - 1);
  cell[1] = (qy & gmask) & ~(w - 1);
  cell[2] = w;
  cell[3] = (int32_t)idx;
  cell[4] = (int32_t)o;
}

constexpr int kMaxBits = 30;

// walk_leaf from the deepest node the point shares with the lane's previous
// descent: that descent's key is pkey, its leaf level plev (0: none) and its
// nodes by depth are in path[d * kBlock].  The top digits the two keys share
// select the same nodes and the same octants, none of them a leaf above
// plev, so the result is walk_leaf's.  Updates pkey, plev and the path.
__device__ inline void walk_leaf_path(float px, float py, int bits,
                                      const int32_t *__restrict__ octree, int64_t size,
                                      int32_t *path, uint64_t &pkey, int &plev, int32_t cell[5]) {
  const int32_t qx = (int32_t)px, qy = (int32_t)py;
  const int64_t c[2] = {qx, qy};
  uint64_t lo, hi;
  morton128<2>(c, bits, lo, hi);
  const uint64_t key = lo & ((1ull << (2 * bits)) - 1);
  int d = 0;
  if (plev > 0) {
    const uint64_t x = key ^ pkey;
    const int common = x ? (__clzll((long long)x) - (64 - 2 * bits)) >> 1 : bits;
    d = common < plev - 1 ? common : plev - 1;
  }
  int64_t idx = path[d * kBlock];
  uint32_t o = 0;
  int32_t lev = d;
  for (int sh = 2 * (bits - d) - 2; sh >= 0; sh -= 2) {
    o = (uint32_t)(lo >> sh) & 3u;
    ++lev;
    const int32_t *node = octree + idx * 5;
    const int32_t child = node[o];
    if ((node[4] >> o) & 1) break;
    if (child < 0 || child >= size) break;
    idx = child;
    path[lev * kBlock] = (int32_t)idx;
  }
  pkey = key;
  plev = lev;
  const int32_t w = (int32_t)(1u << (bits - lev));
  const int32_t gmask = (int32_t)((1u << bits) - 1);
  cell[0] = (qx & gmask) & ~(w - 1);
  cell[1] = (qy & gmask) & ~(w - 1);
  cell[2] = w;
  cell[3] = (int32_t)idx;
  cell[4] = (int32_t)o;
}

// One pass over the segments.  MODE kWalkCount: counts and status;
// kWalkWrite: the cells at offsets[i]; kWalkSpec: counts and status, and
// the first K cells of segment i as records at scratch + K i; kWalkRest: for
// the segments with more than K cells, cells K.. at offsets[i] + K.
//
// A wave takes the segments [w per, (w + 1) per) in turn: a lane whose segment
// has ended takes the next one once kWalkRefill lanes stand idle (segments
// differ in length, and 64 of them take as long as their longest: 2^20
// segments of up to 1/256 of the grid visit 11 cells on average and 30 at
// most).  What bounds it then is the requests: each lane's node words and
// records lie on lines of their own.  A kept cell is one 16-byte record
// (origin x, origin y, parent, octant | level << 2), one store in place of five.
enum { kWalkCount = 0, kWalkWrite = 1, kWalkSpec = 2, kWalkRest = 3 };
#ifndef PGVD_WALK_REFILL
#define PGVD_WALK_REFILL 16
#endif
constexpr uint32_t kWalkRefill = PGVD_WALK_REFILL;

template <int MODE>
__global__ __launch_bounds__(kBlock) void cell_walk_kernel(
    const float *__restrict__ segs, int64_t n, int64_t per, int bits,
    const int32_t *__restrict__ octree, int64_t size, uint32_t *__restrict__ counts,
    int32_t *__restrict__ status, const int64_t *__restrict__ offsets,
    int32_t *__restrict__ cells, int4 *__restrict__ scratch, int K, uint64_t *__restrict__ zero,
    int64_t words) {
  // the scan that follows finds its workspace clear
  if (MODE == kWalkCount || MODE == kWalkSpec)
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < words;
         i += (int64_t)gridDim.x * kBlock)
      zero[i] = 0;
  // each lane's last descent, node per depth (depth 0 is the root)
  __shared__ int32_t s_path[(kMaxBits + 1) * kBlock];
  int32_t *path = s_path + threadIdx.x;
  path[0] = 0;
  const uint32_t wave = blockIdx.x * (kBlock / 64) +
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int64_t next = wave * per;                       // uniform over the wave
  const int64_t end = next + per < n ? next + per : n;
  bool active = false;
  int64_t s = 0;
  float ax = 0, ay = 0, vx = 0, vy = 0, len = 0, ct = 0, cx = 0, cy = 0;
  int dx = 0, dy = 0, count = 0;
  int32_t bcell[5], cell[5] = {0, 0, 1, 0, 0}, ncell[5];
  uint64_t pkey = 0;
  int plev = 0;
  bcell[0] = bcell[1] = 0;
  // The whole wave takes every round, idle lanes included (the ballot counts
  // them): one way back to the loop's head, and scalar conditions for the
  // refill and the end.  A `continue` for the idle lanes would let them turn in
  // a loop of their own, apart from the lanes that still walk.
  for (;;) {
    const uint64_t idle = __ballot(!active);
    const uint32_t nidle = (uint32_t)__popcll(idle);
    if (next >= end && nidle == 64) break;
    if (next < end && nidle >= kWalkRefill) {
      const int64_t mine = next + __popcll(idle & lanemask_lt());
      next += nidle;
      if (!active && mine < end && !(MODE == kWalkRest && counts[mine] <= (uint32_t)K)) {
        s = mine;
        ax = segs[4 * s];
        ay = segs[4 * s + 1];
        const float bx = segs[4 * s + 2], by = segs[4 * s + 3];
        dx = bx > ax ? 1 : (bx < ax ? -1 : 0);
        dy = by > ay ? 1 : (by < ay ? -1 : 0);
        walk_dir(ax, ay, bx, by, vx, vy, len);
        ct = 0.0f;
        cx = ax;
        cy = ay;
        count = 0;
        plev = 0;
        walk_leaf(bx, by, bits, octree, size, bcell);
        walk_leaf_path(cx, cy, bits, octree, size, path, pkey, plev, cell);
        active = true;
      }
    } else if (active) {
      int st = 0;
      bool done = false;
      if (++count > kWalkMax) {
        st = 1;
        --count;
        done = true;
      } else {
        if (MODE == kWalkSpec) {
          if (count <= K)
            scratch[(int64_t)K * s + count - 1] =
                make_int4(cell[0], cell[1], cell[3], cell[4] | plev << 2);
        } else if (MODE == kWalkWrite || (MODE == kWalkRest && count > K)) {
          int32_t *out = cells + 5 * (offsets[s] + count - 1);
#pragma unroll
          for (int k = 0; k < 5; ++k) out[k] = cell[k];
        }
        float ts[4], px[4], py[4];
        const uint32_t keep = walk_isects(ax, ay, vx, vy, len, cell[0], cell[1], cell[2], ts, px, py);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (((keep >> i) & 1) && ts[i] > ct) {
            ct = ts[i];
            cx = px[i];
            cy = py[i];
          }
        if (cx == (float)cell[0] && cx != 0.0f && dx == -1) cx -= 1.0f;
        if (cy == (float)cell[1] && cy != 0.0f && dy == -1) cy -= 1.0f;
        walk_leaf_path(cx, cy, bits, octree, size, path, pkey, plev, ncell);
        done = keep == 0 || (cell[0] == bcell[0] && cell[1] == bcell[1]) ||
               (ncell[0] == cell[0] && ncell[1] == cell[1]);
#pragma unroll
        for (int k = 0; k < 5; ++k) cell[k] = ncell[k];
      }
      if (done) {
        if (MODE == kWalkCount || MODE == kWalkSpec) {
          counts[s] = (uint32_t)count;
          if (status) status[s] = st;
        }
        active = false;
      }
    }
  }
}

// Moves the speculative pass's first min(count, K) cells of every segment
// to their offsets; one thread per (segment, slot), K a power of two.
__global__ __launch_bounds__(kBlock) void walk_compact_kernel(
    const int4 *__restrict__ scratch, const uint32_t *__restrict__ counts,
    const int64_t *__restrict__ offsets, int64_t n, int log2k, int bits,
    int32_t *__restrict__ cells) {
  const int64_t slots = n << log2k;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < slots;
       i += (int64_t)gridDim.x * kBlock) {
    const int64_t s = i >> log2k;
    const uint32_t k = (uint32_t)(i & ((int64_t(1) << log2k) - 1));
    if (k < counts[s]) {
      const int4 r = scratch[i];
      int32_t *dst = cells + 5 * (offsets[s] + k);
      dst[0] = r.x;
      dst[1] = r.y;
      dst[2] = (int32_t)(1u << (bits - (r.w >> 2)));
      dst[3] = r.z;
      dst[4] = r.w & 3;
    }
  }
}

// offsets[0] = 0, offsets[i + 1] = counts[0] + ... + counts[i], of one array
// of counts to each row of the grid; 16 counts a thread, 4096 per tile; ws: word
// 0 tile counter, status array from word 4.  The look-back over the tiles
// bounds it: with 4 counts a thread a refinement of 10,000 loops (two scans of
// 2.2 M counts a build) took 6.46 ms, with 8 6.09, with 16 6.01, and the walks
// of 2^20 segments 918, 910 and 905 us.
constexpr int kWalkScanPer = 16;
__global__ __launch_bounds__(kBlock) void walk_scan_kernel(ScanJob a, ScanJob b, int64_t n) {
  __shared__ uint32_t s_w[kBlock / 64];
  __shared__ int s_tile;
  const ScanJob j = blockIdx.y ? b : a;
  const int t = threadIdx.x;
  if (t == 0) s_tile = (int)atomicAdd(reinterpret_cast<unsigned int *>(j.ws), 1u);
  __syncthreads();
  const int tile = s_tile;
  const int64_t i0 = ((int64_t)tile * kBlock + t) * kWalkScanPer;
  uint32_t c[kWalkScanPer], sum = 0;
  load_run<uint32_t, kWalkScanPer>(
      j.counts + i0, i0 < n ? (uint32_t)min((int64_t)kWalkScanPer, n - i0) : 0u, c);
#pragma unroll
  for (int k = 0; k < kWalkScanPer; ++k) sum += c[k];
  uint32_t total;
  const uint32_t ex = block_excl_sum<uint32_t>(sum, s_w, &total);
  uint64_t run = tile_prefix<kBlock>(j.ws + 4, tile, total) + ex;
  if (tile == 0 && t == 0) j.offsets[0] = 0;
#pragma unroll
  for (int k = 0; k < kWalkScanPer; ++k) {
    run += c[k];
    if (i0 + k < n) j.offsets[i0 + k + 1] = (int64_t)run;
    if (j.total && i0 + k == n - 1) *j.total = run;
  }
}

}  // namespace

constexpr int64_t kWalkScanTile = kWalkScanPer * kBlock;
int64_t walk_scan_ws_words(int64_t n) { return 4 + (n + kWalkScanTile - 1) / kWalkScanTile; }

int walk_log2_kept(int64_t n) {
  int k = 5;
  while (k < 10 && (n << (k + 1)) * 16 <= (int64_t(64) << 20)) ++k;
  return k;
}

// The walk's grid and segments per wave: a wave per 64 segments, up to about 20
// per CU (what the descents' LDS allows), each with its own run of them; and
// where that leaves the chip short of waves, up to 10 per CU with fewer
// segments each, down to 4: a wave then waits for fewer lanes' lines in each
// step (20,000 segments 83.5 -> 76 us, 2,000 77.7 -> 68.5 us; 65,536 and up
// take the same time either way).
static unsigned walk_grid(int64_t n, int64_t *per) {
  const int64_t waves = std::min<int64_t>(
      (n + 3) / 4, std::max<int64_t>(256 * 10, std::min<int64_t>((n + 63) / 64, 256 * 20)));
  *per = (n + waves - 1) / waves;
  return (unsigned)((waves + kBlock / 64 - 1) / (kBlock / 64));
}

void launch_cell_walk_count(const float *segs, int64_t n, int bits, const int32_t *octree,
                            int64_t size, uint32_t *counts, int32_t *status, int64_t *offsets,
                            uint64_t *ws, void *scratch, int log2k, hipStream_t s) {
  int64_t per;
  const unsigned grid = walk_grid(n, &per);
  const int64_t words = walk_scan_ws_words(n);
  if (scratch)
    cell_walk_kernel<kWalkSpec><<<grid, kBlock, 0, s>>>(segs, n, per, bits, octree, size, counts,
                                                        status, nullptr, nullptr,
                                                        static_cast<int4 *>(scratch), 1 << log2k,
                                                        ws, words);
  else
    cell_walk_kernel<kWalkCount><<<grid, kBlock, 0, s>>>(segs, n, per, bits, octree, size, counts,
                                                         status, nullptr, nullptr, nullptr, 0, ws,
                                                         words);
  const ScanJob j{counts, offsets, ws, nullptr};
  launch_offsets_scan(j, j, 1, n, s);
}

void launch_offsets_scan(const ScanJob &a, const ScanJob &b, int jobs, int64_t n, hipStream_t s) {
  const int64_t tiles = (n + kWalkScanTile - 1) / kWalkScanTile;
  if (tiles > 0) walk_scan_kernel<<<dim3((unsigned)tiles, jobs), kBlock, 0, s>>>(a, b, n);
}

void launch_cell_walk_write(const float *segs, int64_t n, int bits, const int32_t *octree,
                            int64_t size, const int64_t *offsets, int32_t *cells,
                            const void *scratch, uint32_t *counts, int log2k, hipStream_t s) {
  int64_t per;
  const unsigned grid = walk_grid(n, &per);
  if (!scratch) {
    cell_walk_kernel<kWalkWrite><<<grid, kBlock, 0, s>>>(segs, n, per, bits, octree, size, nullptr,
                                                         nullptr, offsets, cells, nullptr, 0,
                                                         nullptr, 0);
    return;
  }
  int64_t cgrid = ((n << log2k) + kBlock - 1) / kBlock;
  if (cgrid > 16384) cgrid = 16384;
  walk_compact_kernel<<<(unsigned)cgrid, kBlock, 0, s>>>(static_cast<const int4 *>(scratch), counts,
                                                         offsets, n, log2k, bits, cells);
  cell_walk_kernel<kWalkRest><<<grid, kBlock, 0, s>>>(segs, n, per, bits, octree, size, counts,
                                                      nullptr, offsets, cells, nullptr,
                                                      1 << log2k, nullptr, 0);
}

}  // namespace pgvd
