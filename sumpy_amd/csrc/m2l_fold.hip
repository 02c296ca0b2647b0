// The folded M2L (see m2l_fold.h): plan, class data, packed multipoles and the
// C-ABI.
#include "m2l_fold.h"

namespace sumpyhip {
namespace m2l_fold {

#define DECLARE(NAME)                                                        \
  int m2l_fold_apply_##NAME(int order, const ApplyArgs &a, hipStream_t st);  \
  int m2l_fold_max_wg_##NAME(int order, int *out);
DECLARE(f64) DECLARE(f64a) DECLARE(f64b)
DECLARE(f32) DECLARE(f32a) DECLARE(f32b)
DECLARE(c128) DECLARE(c128a) DECLARE(c128b)
DECLARE(c64) DECLARE(c64a) DECLARE(c64b)
#undef DECLARE

// the instance of a precision, kind and order group
#define BY_GROUP(F, NAME, order, ...)                                            \
  (order <= 8 ? m2l_fold_##F##_##NAME(order, __VA_ARGS__)                        \
   : order <= 10 ? m2l_fold_##F##_##NAME##a(order, __VA_ARGS__)                  \
                 : m2l_fold_##F##_##NAME##b(order, __VA_ARGS__))
#define BY_ORDER(F, order, ...)                                                  \
  (precision == 0 ? (is_complex ? BY_GROUP(F, c128, order, __VA_ARGS__)          \
                                : BY_GROUP(F, f64, order, __VA_ARGS__))          \
                  : (is_complex ? BY_GROUP(F, c64, order, __VA_ARGS__)           \
                                : BY_GROUP(F, f32, order, __VA_ARGS__)))

namespace {

// {{{ plan: target tiles, their class slots and sources

struct PlanArgs {
  int ntgt, nboxes, nlev, ax, maxslots;
  double root_extent;
  const int *target_boxes, *starts, *lists, *classes, *class_code;
  const int *box_levels;
  const double *centers;
  int lev_slot[MAXLEV];     // tree level -> level of the plan, -1: not in it
  int block_base[MAXLEV + 1];
};

// octant (within its parent) of every target box with a list 2
__global__ __launch_bounds__(256) void fold_keys_kernel(PlanArgs a, int *keys) {
  const int i = blockIdx.x*256 + threadIdx.x;
  if (i >= a.ntgt) return;
  const int tb = a.target_boxes[i], lev = a.box_levels[tb];
  const int slot = lev < MAXLEV ? a.lev_slot[lev] : -1;
  int key = 8*a.nlev;
  if (slot >= 0 && a.starts[i + 1] > a.starts[i]) {
    const double h = ldexp(a.root_extent, -lev);
    int oct = 0;
    for (int d = 0; d < 3; ++d) {
      const double *c = a.centers + (size_t)d*a.nboxes;
      const double x = (c[tb] - (c[0] - 0.5*a.root_extent))/h;
      oct |= ((int)floor(x) & 1) << d;
    }
    key = 8*slot + oct;
  }
  keys[i] = key;
}

// position (tile, column) of every sorted target.  Tiles hold 16 targets of
// one octant of one level; tile j of every octant comes before tile j + 1, so
// that consecutive tiles cover one region of space (shared source rows).
__global__ __launch_bounds__(256) void fold_tiles_kernel(PlanArgs a, const int *sorted,
                                                         const long long *order,
                                                         const long long *key_start,
                                                         int *tile_target, int *tgt_pos) {
  const int p = blockIdx.x*256 + threadIdx.x;
  if (p >= a.ntgt) return;
  const int key = sorted[p], i = (int)order[p];
  if (key >= 8*a.nlev) {
    tgt_pos[i] = -1;
    return;
  }
  const int lev = key >> 3, oct = key & 7;
  const int q = p - (int)key_start[key], j = q/TCOL;
  int rank = 0;
  for (int o = 0; o < 8; ++o) {
    const int k = 8*lev + o;
    const int nt = ((int)(key_start[k + 1] - key_start[k]) + TCOL - 1)/TCOL;
    rank += min(nt, j) + (o < oct && nt > j);
  }
  const int pos = (a.block_base[lev]*WAVES + rank)*TCOL + q % TCOL;
  tile_target[pos] = a.target_boxes[i];
  tgt_pos[i] = pos;
}

// canonical vector of a list-2 vector: |n_i| on the folded axes
__device__ __forceinline__ int canonical(int id, int ax) {
  int n[3] = {id/49 - 3, id/7 % 7 - 3, id % 7 - 3};
  for (int d = 0; d < ax; ++d) n[d] = abs(n[d]);
  return (n[0] + 3)*49 + (n[1] + 3)*7 + n[2] + 3;
}

// index of a canonical vector in the class tables: 4 values on a folded axis
// (0..3), 7 on the others
__device__ __host__ __forceinline__ int table_index(int id, int ax) {
  const int n[3] = {id/49, id/7 % 7, id % 7};
  int r = 0;
  for (int d = 0; d < 3; ++d) r = d < ax ? 4*r + n[d] - 3 : 7*r + n[d];
  return r;
}

// sources of every (tile, vector, column) and the tiles of a block that have
// a vector (bits of present)
__global__ __launch_bounds__(256) void fold_sources_kernel(PlanArgs a, const int *tgt_pos,
                                                           int *src, int *present) {
  const int i = blockIdx.x*4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (i >= a.ntgt) return;
  const int pos = tgt_pos[i];
  if (pos < 0) return;
  const int tile = pos/TCOL, col = pos % TCOL, block = tile/WAVES;
  for (int e = a.starts[i] + lane; e < a.starts[i + 1]; e += 64) {
    const int id = a.class_code[a.classes[e]];
    src[((size_t)tile*NVEC + id)*TCOL + col] = a.lists[e];
    atomicOr(&present[(size_t)block*NVEC + canonical(id, a.ax)], 1 << tile % WAVES);
  }
}

// the slots (canonical vector | table index << 16) of every block by type, the
// cost before each of them, the slots up to each type and the block's cost
__global__ __launch_bounds__(64) void fold_slots_kernel(int ax, int maxslots, const int *present,
                                                        int *slots, int *costs, int *type_end,
                                                        long long *block_cost) {
  const int b = blockIdx.x, lane = threadIdx.x;
  int n = 0, sum = 0;
  for (int type = 0; type < 8; ++type) {
    for (int i0 = 0; i0 < NVEC; i0 += 64) {
      const int id = i0 + lane;
      const int zero =
          ((id/49 == 3) | (id/7 % 7 == 3) << 1 | (id % 7 == 3) << 2) & ((1 << ax) - 1);
      const int tiles = id < NVEC && zero == type ? present[(size_t)b*NVEC + id] : 0;
      const unsigned long long m = __ballot(tiles != 0);
      if (m == 0) continue;
      const int at = n + __popcll(m & ((1ull << lane) - 1));
      const int c = tiles ? slot_cost(id, ax) : 0;
      int upto = c;  // inclusive scan over the wave
      for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(upto, o, 64);
        if (lane >= o) upto += t;
      }
      const int total = __shfl(upto, 63, 64);
      if (tiles && at < maxslots) {
        slots[(size_t)b*maxslots + at] = id | table_index(id, ax) << 16;
        costs[(size_t)b*maxslots + at] = sum + upto - c;
      }
      n = min(n + __popcll(m), maxslots);
      sum += total;
    }
    if (lane == 0) type_end[8*b + type] = n;
  }
  if (lane == 0) block_cost[b] = sum;
}

// }}}

// {{{ class data of the canonical vectors

struct LayoutArgs {
  int ax, order, s0, s1, size;
  int base[8];
};

// table[idx][plane][entry]: the class data of canonical vector idx in the LDS
// layout, from the data of class rep[idx] with the signs of the reflection
// sgn[idx] that takes it there (rep < 0: vector not present, left alone)
template <typename T>
__global__ __launch_bounds__(256) void fold_table_kernel(LayoutArgs l, int planes, int M1,
                                                         int M2, int ncirc, const int *rep,
                                                         const int *sgn, const double *data,
                                                         T *table) {
  const int idx = blockIdx.y, cls = rep[idx];
  if (cls < 0) return;
  const int flip = sgn[idx];
  const double *D = data + (size_t)cls*planes*ncirc;
  T *out = table + (size_t)idx*planes*l.size;
  for (int e = blockIdx.x*256 + threadIdx.x; e < planes*l.size; e += gridDim.x*256) {
    const int q = e/l.size, w = e - q*l.size;
    int par = 0;
    while (par + 1 < (1 << l.ax) && w >= l.base[par + 1]) ++par;
    int r = w - l.base[par];
    int m[3];
    m[0] = r/l.s0; r -= m[0]*l.s0;
    m[1] = r/l.s1; m[2] = r - m[1]*l.s1;
    for (int d = 0; d < l.ax; ++d) m[d] = 2*m[d] + (par >> d & 1);
    const bool on = m[0] + m[1] + m[2] <= 2*l.order && m[0] <= 2 && m[1] < M1 && m[2] < M2;
    double x = 0;
    if (on) {
      x = D[(size_t)q*ncirc + ((size_t)m[0]*M1 + m[1])*M2 + m[2]];
      if (__popc(((m[0] & 1) | (m[1] & 1) << 1 | (m[2] & 1) << 2) & flip) & 1) x = -x;
    }
    out[e] = T(x);
  }
}

// }}}

// {{{ multipoles in k order

// packed[box][k] = src[box][kmap[k]] (zero for -1), complex entries as
// (plane, pair) blocks: [kp][lane group][re0, re1, im0, im1]
template <typename T, bool CX>
__global__ __launch_bounds__(256) void fold_pack_kernel(int nboxes, int nstored, int kpad,
                                                        const double *src, const int *kmap,
                                                        T *packed) {
  const size_t n = (size_t)nboxes*kpad;
  for (size_t i = blockIdx.x*(size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x*256) {
    const size_t b = i/kpad;
    const int p = (int)(i - b*kpad), k = kmap[p];
    const bool on = k >= 0;
    if (CX) {
      double2 v = {0, 0};
      if (on) v = reinterpret_cast<const double2 *>(src)[b*nstored + k];
      T *o = packed + b*2*kpad + (size_t)(p >> 1)*4 + (p & 1);
      o[0] = T(v.x);
      o[2] = T(v.y);
    } else {
      packed[i] = on ? T(src[b*nstored + k]) : T(0);
    }
  }
}

// }}}

template <int ORD>
void sizes_of(int *out) {
  for (int p = 0; p < Fold<ORD>::NP; ++p) {
    out[3 + p] = Fold<ORD>::nrb(p);
    out[11 + p] = Fold<ORD>::nkp(p);
  }
  out[0] = Fold<ORD>::AX; out[1] = Fold<ORD>::NRB; out[2] = Fold<ORD>::NKP;
  for (int f64 = 0; f64 < 2; ++f64) {
    int *o = out + 19 + 3*f64;
    o[0] = f64 ? Layout<ORD, true>::S0 : Layout<ORD, false>::S0;
    o[1] = f64 ? Layout<ORD, true>::S1 : Layout<ORD, false>::S1;
    o[2] = f64 ? Layout<ORD, true>::SIZE : Layout<ORD, false>::SIZE;
    for (int d = 0; d < Fold<ORD>::NP; ++d)
      out[25 + 8*f64 + d] = f64 ? Layout<ORD, true>::base(d) : Layout<ORD, false>::base(d);
  }
}

int fill_plan(PlanArgs &p, int ax, int nlevels, const int *lev_slot, int nlev,
              const int *block_base, double root_extent, int nboxes, const int *box_levels,
              const double *centers, int ntgt, const int *target_boxes, const int *starts,
              const int *lists, const int *classes, const int *class_code) {
  SUMPY_REQUIRE(nlevels >= 0 && nlevels <= MAXLEV && nlev >= 1 && nlev <= nlevels,
                "m2l_fold_plan: %d levels (at most %d)", nlevels, MAXLEV);
  SUMPY_REQUIRE(ax >= 0 && ax <= 3, "m2l_fold_plan: %d folded axes", ax);
  p.ntgt = ntgt; p.nboxes = nboxes; p.nlev = nlev; p.ax = ax;
  p.root_extent = root_extent;
  p.target_boxes = target_boxes; p.starts = starts; p.lists = lists;
  p.classes = classes; p.class_code = class_code;
  p.box_levels = box_levels; p.centers = centers;
  for (int l = 0; l < MAXLEV; ++l) p.lev_slot[l] = l < nlevels ? lev_slot[l] : -1;
  for (int l = 0; l <= nlev; ++l) p.block_base[l] = block_base[l];
  return SUMPYHIP_OK;
}

}  // namespace
}  // namespace m2l_fold
}  // namespace sumpyhip

using namespace sumpyhip;
using namespace sumpyhip::m2l_fold;

extern "C" int sumpyhip_m2l_fold_sizes(int order, int *out) {
  SUMPY_REQUIRE(out, "m2l_fold_sizes: null output");
  switch (order) {
    case 1: sizes_of<1>(out); break;
    case 2: sizes_of<2>(out); break;
    case 3: sizes_of<3>(out); break;
    case 4: sizes_of<4>(out); break;
    case 5: sizes_of<5>(out); break;
    case 6: sizes_of<6>(out); break;
    case 7: sizes_of<7>(out); break;
    case 8: sizes_of<8>(out); break;
    case 9: sizes_of<9>(out); break;
    case 10: sizes_of<10>(out); break;
    case 11: sizes_of<11>(out); break;
    case 12: sizes_of<12>(out); break;
    default: return set_error(SUMPYHIP_ENOTIMPL, "m2l_fold: order %d (1..12)", order);
  }
  return SUMPYHIP_OK;
}

extern "C" int sumpyhip_m2l_fold_max_wg(int precision, int is_complex, int order, int *out) {
  SUMPY_REQUIRE(out && (precision == 0 || precision == 1), "m2l_fold_max_wg: bad arguments");
  return BY_ORDER(max_wg, order, out);
}

extern "C" int sumpyhip_m2l_fold_keys(int ax, int nlevels, const int *lev_slot, int nlev,
                                      const int *block_base, double root_extent, int nboxes,
                                      const int *box_levels, const double *centers, int ntgt,
                                      const int *target_boxes, const int *starts, int *keys,
                                      void *stream) {
  PlanArgs p{};
  int rc = fill_plan(p, ax, nlevels, lev_slot, nlev, block_base, root_extent, nboxes,
                     box_levels, centers, ntgt, target_boxes, starts, nullptr, nullptr, nullptr);
  if (rc) return rc;
  if (ntgt == 0) return SUMPYHIP_OK;
  fold_keys_kernel<<<(ntgt + 255)/256, 256, 0, (hipStream_t)stream>>>(p, keys);
  return check_launch("m2l_fold_keys");
}

extern "C" int sumpyhip_m2l_fold_plan(int ax, int nlevels, const int *lev_slot, int nlev,
                                      const int *block_base, double root_extent, int nboxes,
                                      const int *box_levels, const double *centers, int ntgt,
                                      const int *target_boxes, const int *starts,
                                      const int *lists, const int *classes,
                                      const int *class_code, const int *sorted_keys,
                                      const long long *order, const long long *key_start,
                                      int *tile_target, int *tgt_pos, int *src, int *present,
                                      int maxslots, int *slots, int *slot_costs,
                                      int *type_end, long long *block_costs, void *stream) {
  PlanArgs p{};
  int rc = fill_plan(p, ax, nlevels, lev_slot, nlev, block_base, root_extent, nboxes,
                     box_levels, centers, ntgt, target_boxes, starts, lists, classes,
                     class_code);
  if (rc) return rc;
  if (ntgt == 0) return SUMPYHIP_OK;
  hipStream_t st = (hipStream_t)stream;
  fold_tiles_kernel<<<(ntgt + 255)/256, 256, 0, st>>>(p, sorted_keys, order, key_start,
                                                      tile_target, tgt_pos);
  rc = check_launch("m2l_fold_tiles");
  if (rc) return rc;
  fold_sources_kernel<<<(ntgt + 3)/4, 256, 0, st>>>(p, tgt_pos, src, present);
  rc = check_launch("m2l_fold_sources");
  if (rc) return rc;
  const int nblocks = block_base[nlev];
  if (nblocks == 0) return SUMPYHIP_OK;
  fold_slots_kernel<<<nblocks, 64, 0, st>>>(ax, maxslots, present, slots, slot_costs, type_end,
                                              block_costs);
  return check_launch("m2l_fold_slots");
}

extern "C" int sumpyhip_m2l_fold_table(int precision, int is_complex, int order, int ntable,
                                       const int *circ_shape, const int *rep, const int *sgn,
                                       const double *class_data, void *table, void *stream) {
  int sz[41] = {0};
  int rc = sumpyhip_m2l_fold_sizes(order, sz);
  if (rc) return rc;
  SUMPY_REQUIRE(precision == 0 || precision == 1, "m2l_fold_table: precision %d", precision);
  SUMPY_REQUIRE(circ_shape && circ_shape[0] == 3 && circ_shape[1] == 2*order + 1 &&
                    circ_shape[2] == 2*order + 1,
                "m2l_fold_table: class data shape does not match order %d", order);
  if (ntable == 0) return SUMPYHIP_OK;
  const int f64 = precision == 0, planes = is_complex ? 2 : 1;
  LayoutArgs l{};
  l.ax = sz[0]; l.order = order;
  l.s0 = sz[19 + 3*f64]; l.s1 = sz[20 + 3*f64]; l.size = sz[21 + 3*f64];
  for (int d = 0; d < 8; ++d) l.base[d] = sz[25 + 8*f64 + d];
  const int ncirc = circ_shape[0]*circ_shape[1]*circ_shape[2];
  const dim3 grid((planes*l.size + 1023)/1024, ntable);
  hipStream_t st = (hipStream_t)stream;
  if (f64)
    fold_table_kernel<double><<<grid, 256, 0, st>>>(l, planes, circ_shape[1], circ_shape[2],
                                                    ncirc, rep, sgn, class_data,
                                                    (double *)table);
  else
    fold_table_kernel<float><<<grid, 256, 0, st>>>(l, planes, circ_shape[1], circ_shape[2],
                                                   ncirc, rep, sgn, class_data, (float *)table);
  return check_launch("m2l_fold_table");
}

extern "C" int sumpyhip_m2l_fold_pack(int precision, int is_complex, int nboxes, int nstored,
                                      int kpad, const double *src, const int *kmap,
                                      void *packed, void *stream) {
  SUMPY_REQUIRE(precision == 0 || precision == 1, "m2l_fold_pack: precision %d", precision);
  SUMPY_REQUIRE(nboxes >= 0 && nstored > 0 && kpad > 0 && kpad % 8 == 0 && kpad >= nstored,
                "m2l_fold_pack: row of %d coefficients as %d", nstored, kpad);
  if (nboxes == 0) return SUMPYHIP_OK;
  const size_t n = (size_t)nboxes*kpad;
  const int grid = (int)((n + 255)/256 < 16384 ? (n + 255)/256 : 16384);
  hipStream_t st = (hipStream_t)stream;
#define PACK(T, CX) \
  fold_pack_kernel<T, CX><<<grid, 256, 0, st>>>(nboxes, nstored, kpad, src, kmap, (T *)packed)
  if (precision == 0) { if (is_complex) PACK(double, true); else PACK(double, false); }
  else { if (is_complex) PACK(float, true); else PACK(float, false); }
#undef PACK
  return check_launch("m2l_fold_pack");
}

extern "C" int sumpyhip_m2l_fold_apply(int precision, int is_complex, int order, int nblocks,
                                       int maxslots, int box0, int nboxes, int nstored,
                                       const int *tile_target, const int *src,
                                       const int *slots, const int *slot_costs,
                                       const int *type_end, const int *block_level,
                                       const long long *block_cost, const int *rowmap,
                                       const int *off_t, const int *off_s, const void *packed,
                                       const void *table, long long level_stride, int max_wg,
                                       int min_slots, void *partial, double *out,
                                       void *stream) {
  int sz[41] = {0};
  int rc = sumpyhip_m2l_fold_sizes(order, sz);
  if (rc) return rc;
  SUMPY_REQUIRE(precision == 0 || precision == 1, "m2l_fold_apply: precision %d", precision);
  SUMPY_REQUIRE(max_wg >= 1 && min_slots >= 1, "m2l_fold_apply: bad launch shape");
  SUMPY_REQUIRE(nstored == (order + 1)*(order + 1),
                "m2l_fold_apply: %d coefficients at order %d", nstored, order);
  const unsigned long long row = (unsigned long long)sz[2]*8*(is_complex ? 2 : 1)*
                                 (precision == 0 ? 8 : 4);
  SUMPY_REQUIRE((unsigned long long)nboxes*row < (1ull << 31),
                "m2l_fold_apply: %d packed rows exceed 2 GiB", nboxes);
  if (nblocks == 0) return SUMPYHIP_OK;
  ApplyArgs a{};
  a.nblocks = nblocks; a.maxslots = maxslots; a.nstored = nstored; a.box0 = box0;
  a.nboxes = nboxes; a.max_wg = max_wg; a.min_cost = min_slots*MAX_SLOT_COST;
  a.tile_target = tile_target; a.src = src; a.slots = slots; a.slot_cost = slot_costs;
  a.type_end = type_end; a.block_level = block_level; a.block_cost = block_cost; a.rowmap = rowmap;
  a.off_t = off_t; a.off_s = off_s; a.packed = packed; a.table = table;
  a.level_stride = level_stride; a.out = out; a.partial = partial;
  hipStream_t st = (hipStream_t)stream;
  return BY_ORDER(apply, order, a, st);
}
