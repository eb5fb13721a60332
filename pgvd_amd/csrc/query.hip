// query.hip -- batched octree point location: OctreeUtils::FindLeaf
// (OctreeUtils.cpp:18-71), one lane per query point, on an octree as the
// build writes it (nodes of 2^DIM children and a leaf mask).
//
// The key's digits are taken from the top, the octant masked to DIM bits
// (the reference leaves the mask commented out, :37-41, which is wrong below
// the first digit), and the descent stops at the first octant whose leaf bit
// is set.  Each step is two dependent loads from a node (child and leaf
// mask), and below the top levels every lane's load falls on its own line.
//
// Larger batches first build a table of the octree's cells at a fixed depth D
// (find_leaf_table_depth): entry e is where the descent stands after the D
// digits e, either the node to continue from or, when it ended within them,
// its parent, octant, level and status.  A query then starts with one table
// read instead of D levels of node reads; its outputs are the same as those
// of the plain descent.  The entry of a node to continue from also holds the
// node's leaf mask when each of its leaf octants holds the build's -1, so a
// query that ends at level D + 1 (73% of uniform queries in the octree of
// 2^24 uniform points) reads nothing but its entry.  Every read past the
// table takes a 128-byte line for 8 bytes, and those lines bound the kernel:
// 2^24 random queries in that octree took 798 us with 8-byte entries that
// held only the node, 460 us with the mask in 4-byte entries.
#include <type_traits>

#include "kernels.hpp"

namespace pgvd {

namespace {

// Digit (DIM bits) of the 128-bit key (lo, hi) at bit sh.
template <int DIM>
__device__ inline uint32_t key_digit(uint64_t lo, uint64_t hi, int sh) {
  uint64_t v;
  if (sh >= 64) v = hi >> (sh - 64);
  else if (sh == 0) v = lo;
  else v = (lo >> sh) | (hi << (64 - sh));
  return (uint32_t)v & ((1u << DIM) - 1);
}

// Where the descent stands after the table's D digits.
struct TabCell {
  int32_t idx = 0;       // node to continue from, or the parent where it ended
  uint32_t mask = 0;     // its leaf octants, when all of them hold -1 (else 0)
  bool done = false;     // ended within D digits, at:
  bool plain = false;    // its data is -1
  int32_t level = 0;
  uint32_t octant = 0, status = 0;
};

// Entries of 32 bits for octrees of at most 2^23 nodes, of 64 bits for
// larger ones.  A narrow entry holds idx (bits 0-22) and, while the descent
// goes on, the mask (23-30); where it ended bit 31 is set, and with it the
// status (30: 2 or 0), plain (29) and (level - 1) NC + octant (23-28).
constexpr int64_t kTabNarrowNodes = int64_t(1) << 23;
constexpr uint32_t kTabDone = 1u << 31;

template <int DIM>
__device__ inline uint32_t tab_encode(const TabCell &c, uint32_t *) {
  if (!c.done) return (uint32_t)c.idx | c.mask << 23;
  const uint32_t at = (uint32_t)((c.level - 1) << DIM) | c.octant;
  return kTabDone | (uint32_t)c.idx | at << 23 | (uint32_t)c.plain << 29 |
         (uint32_t)(c.status != 0) << 30;
}
template <int DIM>
__device__ inline TabCell tab_decode(uint32_t e) {
  TabCell c;
  c.idx = (int32_t)(e & 0x7fffffu);
  c.done = (e & kTabDone) != 0;
  if (!c.done) {
    c.mask = (e >> 23) & 0xffu;
  } else {
    const uint32_t at = (e >> 23) & 0x3fu;
    c.level = (int32_t)(at >> DIM) + 1;
    c.octant = at & ((1u << DIM) - 1);
    c.plain = (e >> 29) & 1u;
    c.status = (e >> 30) & 1u ? 2u : 0u;
  }
  return c;
}
template <int DIM>
__device__ inline uint2 tab_encode(const TabCell &c, uint2 *) {
  const uint32_t m = c.done ? kTabDone | (uint32_t)c.level | c.octant << 8 | c.status << 12 |
                                  (uint32_t)c.plain << 16
                            : c.mask;
  return make_uint2((uint32_t)c.idx, m);
}
template <int DIM>
__device__ inline TabCell tab_decode(uint2 e) {
  TabCell c;
  c.idx = (int32_t)e.x;
  c.done = (e.y & kTabDone) != 0;
  if (!c.done) {
    c.mask = e.y;
  } else {
    c.level = (int32_t)(e.y & 0xffu);
    c.octant = (e.y >> 8) & 0xfu;
    c.status = (e.y >> 12) & 0xfu;
    c.plain = (e.y >> 16) & 1u;
  }
  return c;
}

// Builds the depth-D table: one lane per cell e (its D digits, most
// significant first), the same descent as find_leaf_kernel stopped after D
// levels.
template <int DIM, typename E>
__global__ __launch_bounds__(kBlock) void find_leaf_table_kernel(
    const int32_t *__restrict__ octree, int64_t octree_size, int D, E *__restrict__ table) {
  constexpr int NC = 1 << DIM, STRIDE = NC + 1;
  const int64_t cells = int64_t(1) << (D * DIM);
  for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < cells;
       e += (int64_t)gridDim.x * kBlock) {
    int64_t idx = 0;
    TabCell c;
    for (int l = 1; l <= D; ++l) {
      const uint32_t o = (uint32_t)(e >> ((D - l) * DIM)) & (NC - 1);
      const int32_t *node = octree + idx * STRIDE;
      const int32_t child = node[o];
      const bool leaf = (node[NC] >> o) & 1;
      if (leaf || child < 0 || child >= octree_size) {
        c.done = true;
        c.plain = leaf && child == -1;
        c.level = l;
        c.octant = o;
        c.status = leaf ? 0u : 2u;
        break;
      }
      idx = child;
    }
    c.idx = (int32_t)idx;
    if (!c.done) {
      const int32_t *node = octree + idx * STRIDE;
      const uint32_t leaves = (uint32_t)node[NC] & ((1u << NC) - 1);
      uint32_t empty = 0;
#pragma unroll
      for (int o = 0; o < NC; ++o) empty |= (uint32_t)(node[o] == -1) << o;
      c.mask = (leaves & ~empty) == 0 ? leaves : 0u;
    }
    table[e] = tab_encode<DIM>(c, (E *)nullptr);
  }
}

// The top D digits of the key (lo, hi), D * DIM <= 21, starting at bit sh.
__device__ inline uint32_t key_bits(uint64_t lo, uint64_t hi, int sh, int width) {
  uint64_t v;
  if (sh >= 64) v = hi >> (sh - 64);
  else if (sh == 0) v = lo;
  else v = (lo >> sh) | (hi << (64 - sh));
  return (uint32_t)v & ((1u << width) - 1);
}

// E: the table's entries (void: no table).  The queries and the outputs are
// read and written once, past the caches, which then keep more of the table
// and the octree.
template <int DIM, typename E>
__global__ __launch_bounds__(kBlock) void find_leaf_kernel(
    const int32_t *__restrict__ pts, int64_t q, int bits, const int32_t *__restrict__ octree,
    int64_t octree_size, const E *__restrict__ table, int D, int32_t *__restrict__ parent,
    int32_t *__restrict__ octant, int32_t *__restrict__ data, int32_t *__restrict__ level,
    uint32_t *__restrict__ status) {
  constexpr int NC = 1 << DIM, STRIDE = NC + 1;
  constexpr bool TABLE = !std::is_same<E, void>::value;
  const int mbits = bits * DIM;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < q;
       i += (int64_t)gridDim.x * kBlock) {
    int64_t c[DIM];
#pragma unroll
    for (int k = 0; k < DIM; ++k) c[k] = __builtin_nontemporal_load(pts + i * DIM + k);
    uint64_t lo, hi;
    morton128<DIM>(c, bits, lo, hi);
    int64_t idx = 0;
    uint32_t o = 0, st = 1;
    int32_t d = -1, lev = 0;
    int sh0 = mbits - DIM;
    if constexpr (TABLE) {
      const int top = mbits - D * DIM;
      const TabCell t = tab_decode<DIM>(table[key_bits(lo, hi, top, D * DIM)]);
      idx = t.idx;
      if (t.done) {
        lev = t.level;
        o = t.octant;
        st = t.status;
        if (st == 0 && !t.plain) d = octree[idx * STRIDE + o];
        sh0 = -1;
      } else {
        lev = D;
        o = key_digit<DIM>(lo, hi, top);
        sh0 = top - DIM;
        const uint32_t next = sh0 >= 0 ? key_digit<DIM>(lo, hi, sh0) : 0u;
        if (sh0 >= 0 && ((t.mask >> next) & 1u)) {   // a leaf whose data is -1
          o = next;
          lev = D + 1;
          st = 0;
          sh0 = -1;
        }
      }
    }
    for (int sh = sh0; sh >= 0; sh -= DIM) {
      o = key_digit<DIM>(lo, hi, sh);
      ++lev;
      const int32_t *node = octree + idx * STRIDE;
      const int32_t child = node[o];
      if ((node[NC] >> o) & 1) {
        d = child;
        st = 0;
        break;
      }
      if (child < 0 || child >= octree_size) {   // not an octree the build wrote
        st = 2;
        break;
      }
      idx = child;
    }
    __builtin_nontemporal_store((int32_t)idx, parent + i);
    __builtin_nontemporal_store((int32_t)o, octant + i);
    __builtin_nontemporal_store(d, data + i);
    __builtin_nontemporal_store(lev, level + i);
    if (status) __builtin_nontemporal_store(st, status + i);
  }
}

template <int DIM, typename E>
void launch_find_leaf_as(const int32_t *pts, int64_t q, int bits, const int32_t *octree,
                         int64_t octree_size, E *table, int D, int32_t *parent, int32_t *octant,
                         int32_t *data, int32_t *level, uint32_t *status, hipStream_t s) {
  int64_t grid = (q + kBlock - 1) / kBlock;
  if (grid > 8192) grid = 8192;
  if (grid < 1) grid = 1;
  if constexpr (!std::is_same<E, void>::value) {
    const unsigned tgrid = (unsigned)(((int64_t(1) << (D * DIM)) + kBlock - 1) / kBlock);
    find_leaf_table_kernel<DIM, E><<<tgrid, kBlock, 0, s>>>(octree, octree_size, D, table);
  }
  find_leaf_kernel<DIM, E><<<(unsigned)grid, kBlock, 0, s>>>(pts, q, bits, octree, octree_size,
                                                             table, D, parent, octant, data,
                                                             level, status);
}

template <int DIM>
void launch_find_leaf_dim(const int32_t *pts, int64_t q, int bits, const int32_t *octree,
                          int64_t octree_size, void *table, int D, int32_t *parent,
                          int32_t *octant, int32_t *data, int32_t *level, uint32_t *status,
                          hipStream_t s) {
  if (D <= 0)
    launch_find_leaf_as<DIM, void>(pts, q, bits, octree, octree_size, nullptr, 0, parent, octant,
                                   data, level, status, s);
  else if (octree_size <= kTabNarrowNodes)
    launch_find_leaf_as<DIM>(pts, q, bits, octree, octree_size, static_cast<uint32_t *>(table), D,
                             parent, octant, data, level, status, s);
  else
    launch_find_leaf_as<DIM>(pts, q, bits, octree, octree_size, static_cast<uint2 *>(table), D,
                             parent, octant, data, level, status, s);
}

}  // namespace

// The table's depth for q queries: the deepest whose cells number at most q
// (a table costs a few reads per cell), at most four per octree node (past
// that most cells share a node and the table only falls out of the caches:
// 2^24 queries in the octree of 300,000 3D points took 250 us from 2^21
// cells and 210 us from 2^18) and at most 2^kFindLeafTableBits (in the
// octree of 2^24 points 2^24 cells took 568 us, 2^21 460 us).  Below 2^18
// queries the second launch costs what the table saves (100,000 queries: 14
// against 12 us).
int find_leaf_table_depth(int64_t q, int dim, int bits, int64_t octree_size) {
  if (q < (int64_t(1) << 18)) return 0;
  int D = std::min(kFindLeafTableBits / dim, bits);
  while (D > 0 && (int64_t(1) << (D * dim)) > std::min(q, 4 * octree_size)) --D;
  return D;
}

void launch_find_leaf(const int32_t *pts, int64_t q, int dim, int bits, const int32_t *octree,
                      int64_t octree_size, void *table, int D, int32_t *parent, int32_t *octant,
                      int32_t *data, int32_t *level, uint32_t *status, hipStream_t s) {
  if (dim == 2)
    launch_find_leaf_dim<2>(pts, q, bits, octree, octree_size, table, D, parent, octant, data,
                            level, status, s);
  else
    launch_find_leaf_dim<3>(pts, q, bits, octree, octree_size, table, D, parent, octant, data,
                            level, status, s);
}

}  // namespace pgvd
