// Multipole-to-local translation folded by the reflection symmetry of the
// kernel, for octree levels (list-2 vectors n h with integer n, |n_i| <= 3).
//
// The class matrix of a radial kernel obeys A_{Rn} = S_R A_n S_R with S_R the
// diagonal matrix of the signs (-1)^(R . m) of a reflection R of some axes, so
// the sources at the reflections Rn of one vector n share one product:
//   sum_R S_R A_n S_R X_R [t] = sum_s A_n[t, s] Xh_{par(t) ^ par(s)}[s],
//   Xh_d[s] = sum_R (-1)^popc(R & d) X_R[s],
// par(m) the parities of the folded components of a multi-index.  Folding all
// three axes leaves 56 products per target instead of 189, and a vector
// with n_i = 0 has no entries where par(t) ^ par(s) is odd in i, which halves
// its product: 39.5 whole products.  The price is the Walsh-Hadamard transform
// Xh of the sources (m 2^m additions per coefficient for m axes with n_i != 0)
// and rows and columns sorted by parity, each parity class padded to whole
// MFMA blocks.  Low orders fold fewer axes, where the padding
// would cost more than the fold saves (Fold::AX).
//
// Reference pipeline: sumpy/fmm.py:777-920, sumpy/e2e.py:310-558.
#pragma once

#include <type_traits>

#include "common.h"

namespace sumpyhip {
namespace m2l_fold {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));

constexpr int WAVES = 4;       // target tiles of 16 columns per block
constexpr int TCOL = 16;       // target boxes per tile
constexpr int NVEC = 343;      // list-2 vectors, (n_x + 3) 49 + (n_y + 3) 7 + n_z + 3
constexpr int MAXLEV = 32;

// Parity classes, row blocks (16 rows) and k pairs (2 MFMA k steps, 8
// coefficients) of the PDE-compressed set (m_x <= 1) of one order.  A parity
// class is bit 0: m_x, bit 1: m_y, bit 2: m_z (folded axes only).
template <int ORD>
struct Fold {
  // products x padded rows x padded columns per target, by folded axes
  // (0, 1, 2, 3): p = 3: 48k, 86k; p = 5: 363k, 216k, 239k, 323k; p = 7:
  // 774k, 648k, 384k, 485k; p = 8: 1597k, 950k, 718k, 607k
  static constexpr int AX = ORD <= 3 ? 0 : ORD <= 5 ? 1 : ORD <= 7 ? 2 : 3;
  static constexpr int NP = 1 << AX;
  static constexpr int count(int par) {
    int n = 0;
    for (int a = 0; a <= (ORD > 0 ? 1 : 0); ++a)
      for (int b = 0; a + b <= ORD; ++b)
        for (int c = 0; a + b + c <= ORD; ++c)
          if ((((a & 1) | (b & 1) << 1 | (c & 1) << 2) & (NP - 1)) == par) ++n;
    return n;
  }
  static constexpr int nrb(int par) { return (count(par) + 15)/16; }
  static constexpr int nkp(int par) { return (count(par) + 7)/8; }
  static constexpr int rb0(int par) { return par ? rb0(par - 1) + nrb(par - 1) : 0; }
  static constexpr int kp0(int par) { return par ? kp0(par - 1) + nkp(par - 1) : 0; }
  static constexpr int NRB = rb0(NP - 1) + nrb(NP - 1);
  static constexpr int NKP = kp0(NP - 1) + nkp(NP - 1);
  static constexpr int par_of_rb(int rb) {
    int p = 0;
    while (rb >= rb0(p) + nrb(p)) ++p;
    return p;
  }
  // parity class of a k pair
  static constexpr int par_of(int kp) {
    int p = 0;
    while (kp >= kp0(p) + nkp(p)) ++p;
    return p;
  }
};

// f(0), f(1), ..., f(N - 1) with the index a compile-time constant
template <int N, int I = 0, class Fn>
__device__ __forceinline__ void static_for(Fn &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

// Class data of one vector in LDS: the derivatives by parity of their folded
// components, halved there, so that the entry of (t, s) sits at
//   base(par_t ^ par_s) + carry(par_t & par_s) + off(t) + off(s),
// off(m) = S0 q_x + S1 q_y + q_z, q = m >> 1 on folded axes, m on the others;
// the first two terms are instruction immediates.  S1 spreads the 16 rows of
// an MFMA over the LDS banks: by enumeration over S1 < 40, the gathers then
// take at most 1.8 times the conflict-free cycles (FP64, 16 lanes a cycle;
// order 10: 1.78, order 8: 1.13) and 1.9 times (FP32, 32 lanes; order 10:
// 1.51).
template <int ORD, bool F64>
struct Layout {
  typedef Fold<ORD> F;
  static constexpr int S1_64[13] = {0, 3, 6, 7, 10, 11, 22, 22, 10, 10, 20, 14, 14};
  static constexpr int S1_32[13] = {0, 3, 6, 9, 27, 19, 14, 20, 20, 27, 27, 19, 19};
  static constexpr int S1 = F64 ? S1_64[ORD] : S1_32[ORD];
  static constexpr int EY = F::AX >= 2 ? ORD : 2*ORD, EZ = F::AX >= 3 ? ORD : 2*ORD;
  static constexpr int SPAN = S1*EY + EZ + 1, S0 = SPAN;
  static constexpr int planes(int d) { return F::AX == 0 ? 3 : d & 1 ? 1 : 2; }
  static constexpr int base(int d) { return d ? base(d - 1) + planes(d - 1)*SPAN : 0; }
  static constexpr int carry(int c) { return (c & 1 ? S0 : 0) + (c & 2 ? S1 : 0) + (c & 4 ? 1 : 0); }
  // entries, in whole 16-byte vectors
  static constexpr int SIZE = (base(F::NP - 1) + planes(F::NP - 1)*SPAN + 3)/4*4;
};

template <typename T>
struct Mfma;
// operand layouts (checked on gfx950): A[i][k] in lane i + 16k, B[k][j] in
// lane j + 16k; accumulator register r of lane l holds column l % 16 and row
// (l/16) + 4r for the FP64 instruction, 4(l/16) + r for the FP32 one
template <>
struct Mfma<double> {
  typedef v4d acc_t;
  typedef double2 vec2;
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4*r; }
};
template <>
struct Mfma<float> {
  typedef v4f acc_t;
  typedef float2 vec2;
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4*(lane >> 4) + r; }
};

// {{{ the contraction

struct ApplyArgs {
  int nblocks, maxslots, nstored, box0, nboxes, max_wg, min_cost;
  const int *tile_target, *src, *slots, *slot_cost, *type_end, *block_level;
  const long long *block_cost;       // nblocks + 1: cost before each block
  const int *rowmap, *off_t, *off_s;  // off(m) of the padded rows and columns
  const void *packed, *table;
  long long level_stride;            // entries of one level's table
  double *out;                       // one row of nstored (complex) values per box from box0 on
  void *partial;                     // 2 max_wg x WAVES tiles of accumulators
};

// The slots of a block are sorted by type, the set of folded axes with n_i = 0
// (type_end[8 b + z]: slots of block b of the types up to z; type 7 is the
// target itself and has none).  The slots of all blocks in block order lie on one line of cost (slot_cost:
// cost before a slot within its block); workgroup g of G takes the slots that
// begin in [C g/G, C (g+1)/G), so every workgroup does the same work whatever
// the blocks' sizes.  A block whose slots lie in several workgroups is summed
// from their partial accumulators by fold_reduce_kernel.  G leaves a workgroup
// at least MAX_SLOT_COST, so each of them finds a slot.
constexpr int MAX_SLOT_COST = 20;

// cost of a slot: its products (16 at most, halved by every zero component)
// and 4 for the rest.  The tiles of a block keep pace, so a slot costs the same
// however many of them have a source (by their number, the sphere's Helmholtz
// M2L at order 12 took 1334 us, this way 908 us).
__device__ __forceinline__ int slot_cost(int id, int ax) {
  const int n[3] = {id/49, id/7 % 7, id % 7};
  int w = 16;
  for (int d = 0; d < ax; ++d)
    if (n[d] == 3) w >>= 1;
  return w + 4;
}

__device__ __forceinline__ long long num_wg(const ApplyArgs &a, long long cost) {
  const long long g = cost/a.min_cost;
  return g < 1 ? 1 : g > a.max_wg ? a.max_wg : g;
}

// first cost of workgroup g of G
__device__ __forceinline__ long long wg_cost(long long cost, long long g, long long G) {
  return cost*g/G;
}

// workgroup whose range holds cost position c
__device__ __forceinline__ long long wg_of(long long cost, long long c, long long G) {
  long long g = c*G/cost;
  while (g + 1 < G && wg_cost(cost, g + 1, G) <= c) ++g;
  while (g > 0 && wg_cost(cost, g, G) > c) --g;
  return g;
}

// uniform reads through the scalar cache
typedef const __attribute__((address_space(4))) int *ConstInt;

// last block that begins at or before cost position c
__device__ __forceinline__ int block_of(const ApplyArgs &a, long long c) {
  int lo = 0, hi = a.nblocks;
  while (hi - lo > 1) {
    const int mid = (lo + hi)/2;
    if (a.block_cost[mid] <= c) lo = mid; else hi = mid;
  }
  return lo;
}

// first slot of a block that begins at or after cost c within the block
__device__ __forceinline__ int slot_of(const int *cost, int n, long long c) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi)/2;
    if (cost[mid] < c) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// N 4-byte words at byte offset voff + soff of the rows; 0 past the end
template <int N>
struct BufLoad;
template <>
struct BufLoad<2> {
  typedef unsigned type __attribute__((ext_vector_type(2)));
  static __device__ __forceinline__ type get(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
  }
};
template <>
struct BufLoad<4> {
  typedef u4 type;
  static __device__ __forceinline__ type get(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
  }
};

// One wave per tile of 16 targets: all row blocks of the tile accumulate in
// registers.  Per slot (one canonical vector) and k pair, a lane loads 2
// coefficients of each of the vector's sources (B layout: column lane % 16,
// coefficients 2 (lane/16), +1 of the pair; an absent source is past the
// buffer's end and reads as zero), transforms them, and multiplies them by the
// A fragments, gathered from the slot's class data in LDS (double buffered,
// shared by the block's waves; one barrier per slot).  Every slot type has a
// loop of its own, without the products and the transform that its zero
// components leave out.  The sources are fetched DEPTH k pairs ahead.  The k
// pairs are unrolled, so that their buffers are registers and every LDS offset
// but the row's and the column's is immediate (complex FP64: the parity
// classes only; its code would take minutes to compile).
//
// In FP32 the transform adds up to three roundings per source; the long sums of a
// workgroup weigh more, so that the caller keeps its ranges short (their sums are
// added in FP64): the locals are then no further from FP64 than the class
// matrices'.
//
// Bound: issue of the SIMD.  On gfx950 FP64 and FP32 MFMAs do not overlap with
// VALU instructions, of other waves either (measured: 8000 FP64 MFMAs 229 us,
// 128000 additions 507 us, both from two waves of a SIMD 729 us), so the
// transform's additions and the address additions count in full.
template <typename T, int ORD, bool CX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CX && sizeof(T) == 8 ? 1 : 2)))
void fold_apply_kernel(ApplyArgs a) {
  typedef Fold<ORD> F;
  typedef Layout<ORD, sizeof(T) == 8> L;
  typedef typename Mfma<T>::acc_t acc_t;
  typedef typename Mfma<T>::vec2 vec2;
  constexpr int PL = CX ? 2 : 1, AX = F::AX, NP = F::NP, NRB = F::NRB, NKP = F::NKP;
  constexpr int DEPTH = CX || sizeof(T) == 8 || NKP < 2 ? 1 : 2;
  constexpr bool ROLLED = CX && sizeof(T) == 8;
  constexpr int NTYPES = AX == 3 ? 7 : NP;
  constexpr int V16 = PL*L::SIZE*(int)sizeof(T)/16, NV = (V16 + 255)/256;
  constexpr int PART = (NV + NP - 1)/NP;                  // vectors staged per parity class
  constexpr int NPARTS = (NV + PART - 1)/PART;
  constexpr unsigned ROWB = NKP*8*PL*sizeof(T);           // bytes of a packed row
  typedef BufLoad<(int)sizeof(vec2)/4> Load;
  extern __shared__ __align__(16) unsigned char lds[];
  T *sD = reinterpret_cast<T *>(lds);                     // [2][PL][L::SIZE]
  int2 *sK = reinterpret_cast<int2 *>(lds + 2*PL*L::SIZE*sizeof(T));  // [NKP][4]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kg = lane >> 4;
  const long long cost = a.block_cost[a.nblocks];
  const long long G = num_wg(a, cost);
  // consecutive block ids go to different XCDs: give an XCD a contiguous range
  const int per = (a.max_wg + 7)/8;
  const long long g = (long long)(blockIdx.x & 7)*per + (blockIdx.x >> 3);
  if (g >= G) return;
  const long long c_begin = wg_cost(cost, g, G), c_end = wg_cost(cost, g + 1, G);
  const __amdgpu_buffer_rsrc_t X = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void *>(a.packed), 0, (int)((unsigned)a.nboxes*ROWB), 0x00027000);
  constexpr unsigned ABSENT = 0x80000000u;                // (rows are below 2 GiB)
  for (int i = tid; i < NKP*4; i += 256)
    sK[i] = int2{a.off_s[2*i]*(int)sizeof(T), a.off_s[2*i + 1]*(int)sizeof(T)};
  int offT[NRB];             // bytes, as sK
  #pragma unroll
  for (int r = 0; r < NRB; ++r) offT[r] = a.off_t[16*r + col]*(int)sizeof(T);

  for (int b = __builtin_amdgcn_readfirstlane(block_of(a, c_begin));
       b < a.nblocks && a.block_cost[b] < c_end; ++b) {
    const long long cb = a.block_cost[b];
    const ConstInt type_end = (ConstInt)(a.type_end + 8*b);
    const int nsl = type_end[7];
    const int *costs = a.slot_cost + (size_t)b*a.maxslots;
    const int s0 = __builtin_amdgcn_readfirstlane(slot_of(costs, nsl, c_begin - cb));
    const int s1 = __builtin_amdgcn_readfirstlane(slot_of(costs, nsl, c_end - cb));
    if (s0 >= s1) continue;
    const ConstInt slots = (ConstInt)(a.slots + (size_t)b*a.maxslots);
    const int tile = b*WAVES + wave;
    const int *tsrc = a.src + (size_t)tile*NVEC*TCOL + col;
    const T *tab = static_cast<const T *>(a.table) + (size_t)a.block_level[b]*a.level_stride;

    acc_t acc[PL][NRB];
    #pragma unroll
    for (int q = 0; q < PL; ++q)
      #pragma unroll
      for (int r = 0; r < NRB; ++r) acc[q][r] = acc_t{0, 0, 0, 0};

    // this lane's column: source box per reflection of the slot's vector
    auto sources = [&](int id, int (&sb)[NP]) {
      const int c[3] = {id/49 - 3, id/7 % 7 - 3, id % 7 - 3};
      static_for<NP>([&](auto R) {
        sb[R] = tsrc[(id - (R & 1 ? 98*c[0] : 0) - (R & 2 ? 14*c[1] : 0) -
                      (R & 4 ? 2*c[2] : 0))*TCOL];
      });
    };
    // their rows' byte offsets (an axis without a component has one
    // reflection only); whether any column of the tile has one
    auto offsets = [&](const int (&sb)[NP], int id, unsigned (&off)[NP]) {
      const int zero = (id/49 == 3) | (id/7 % 7 == 3) << 1 | (id % 7 == 3) << 2;
      bool on = false;
      static_for<NP>([&](auto R) {
        const bool has = sb[R] >= 0 && (R & zero) == 0;
        off[R] = has ? (unsigned)(sb[R] - a.box0)*ROWB + kg*(unsigned)(2*PL*sizeof(T)) : ABSENT;
        on = on || has;
      });
      return __ballot(on) != 0;
    };
    vec2 x[DEPTH][NP][PL];
    auto load_x = [&](auto skip, int buf, int kp, const unsigned (&off)[NP]) {
      static_for<NP>([&](auto Rc) {
        constexpr int R = Rc;
        if constexpr (!(R & skip)) {
          #pragma unroll
          for (int q = 0; q < PL; ++q)
            x[buf][R][q] = __builtin_bit_cast(
                vec2, Load::get(X, off[R] + q*(unsigned)sizeof(vec2), kp*8*PL*(int)sizeof(T)));
        }
      });
    };
    u4 dreg[PART];
    auto load_d = [&](const T *data, int part) {
      #pragma unroll
      for (int i = 0; i < PART; ++i) {
        const int e = tid + 256*(part*PART + i);
        dreg[i] = reinterpret_cast<const u4 *>(data)[e < V16 ? e : V16 - 1];
      }
    };
    auto store_d = [&](int buf, int part) {
      #pragma unroll
      for (int i = 0; i < PART; ++i) {
        const int e = tid + 256*(part*PART + i);
        if (e < V16) reinterpret_cast<u4 *>(sD + buf*PL*L::SIZE)[e] = dreg[i];
      }
    };
    constexpr std::integral_constant<int, 0> all{};
    int sb[NP];
    unsigned off[NP];
    const int first = slots[s0];
    sources(first & 0xffff, sb);
    bool cur = offsets(sb, first & 0xffff, off);
    __syncthreads();   // the previous segment is done with sD (and sK is written)
    {
      const T *data = tab + (size_t)(first >> 16)*PL*L::SIZE;
      for (int p = 0; p < NPARTS; ++p) {
        load_d(data, p);
        store_d(0, p);
      }
    }
    static_for<DEPTH>([&](auto d) { load_x(all, d, d, off); });
    __syncthreads();
    int buf = 0, slot = s0;
    int2 ko_next = sK[kg];

    static_for<NTYPES>([&](auto zc) {
      constexpr int zero = zc;
      const int end = min(s1, (int)type_end[zero]);
      for (; slot < end; ++slot) {
        const int next = slots[slot + 1 < s1 ? slot + 1 : slot];
        const T *data = tab + (size_t)(next >> 16)*PL*L::SIZE;
        const unsigned char *D = lds + buf*PL*L::SIZE*(int)sizeof(T);
        const bool on = cur;   // slots without a source for this tile: no products
        // one k pair: kp of parity class ps, sources in buffer xb
        auto k_pair = [&](auto psc, auto xbc, int kp) {
          constexpr int ps = psc, xb = xbc;
          const int2 ko = ko_next;
          ko_next = sK[(kp + 1 < NKP ? kp + 1 : 0)*4 + kg];
          vec2 xh[NP][PL];
          static_for<NP>([&](auto Rc) {
            constexpr int R = Rc;
            if constexpr (!(R & zero)) {
              #pragma unroll
              for (int q = 0; q < PL; ++q) xh[R][q] = x[xb][R][q];
            }
          });
          static_for<AX>([&](auto ic) {
            constexpr int bit = 1 << ic;
            static_for<NP>([&](auto Rc) {
              constexpr int R = Rc;
              if constexpr (!(bit & zero) && !(R & (bit | zero))) {
                #pragma unroll
                for (int q = 0; q < PL; ++q) {
                  const vec2 p = xh[R][q], m = xh[R | bit][q];
                  xh[R][q] = vec2{p.x + m.x, p.y + m.y};
                  xh[R | bit][q] = vec2{p.x - m.x, p.y - m.y};
                }
              }
            });
          });
          if (kp + DEPTH == NKP) cur = offsets(sb, next & 0xffff, off);
          if constexpr (ROLLED)
            load_x(all, xb, kp + 1 < NKP ? kp + 1 : 0, off);
          else if (kp + DEPTH < NKP)
            load_x(zc, xb, kp + DEPTH, off);
          else
            load_x(all, xb, xb, off);
          if (on) {
            static_for<2>([&](auto vc) {
              constexpr int v = vc;
              const int kb = v ? ko.y : ko.x;
              static_for<NRB>([&](auto rc) {
                constexpr int rb = rc, pr = F::par_of_rb(rb), d = pr ^ ps;
                constexpr int imm = L::base(d) + L::carry(pr & ps);
                if constexpr (!(d & zero)) {
                  const T xr = v ? xh[d][0].y : xh[d][0].x;
                  const T *A = reinterpret_cast<const T *>(D + (offT[rb] + kb));
                  const T ar = A[imm];
                  acc[0][rb] = Mfma<T>::mma(ar, xr, acc[0][rb]);
                  if constexpr (CX) {
                    const T xi = v ? xh[d][1].y : xh[d][1].x;
                    const T ai = A[imm + L::SIZE];
                    acc[1][rb] = Mfma<T>::mma(ar, xi, acc[1][rb]);
                    acc[0][rb] = Mfma<T>::mma(ai, -xi, acc[0][rb]);
                    acc[1][rb] = Mfma<T>::mma(ai, xr, acc[1][rb]);
                  }
                }
              });
              // keep the scheduler within a k step: what it would hoist costs
              // more registers than there are
              __builtin_amdgcn_sched_barrier(0);
            });
          }
        };
        auto stage = [&](int ps) {
          if (ps > 0 && ps <= NPARTS) store_d(buf ^ 1, ps - 1);
          if (ps < NPARTS) load_d(data, ps);
        };
        if constexpr (ROLLED) {
          static_for<NP>([&](auto ps) {
            stage(ps);
            if (ps == NP - 1) sources(next & 0xffff, sb);
            #pragma unroll 1
            for (int j = 0; j < F::nkp(ps); ++j) k_pair(ps, all, F::kp0(ps) + j);
          });
        } else {
          static_for<NKP>([&](auto kp) {
            constexpr int ps = F::par_of(kp);
            if (kp == F::kp0(ps)) stage(ps);
            if (kp == (NKP > DEPTH + 2 ? NKP - DEPTH - 2 : 0)) sources(next & 0xffff, sb);
            k_pair(std::integral_constant<int, ps>{}, std::integral_constant<int, kp % DEPTH>{},
                   kp);
          });
        }
        if (NPARTS == NP) store_d(buf ^ 1, NP - 1);
        __syncthreads();
        buf ^= 1;
      }
    });

    if (s0 == 0 && s1 == nsl) {
      const int tb = a.tile_target[(size_t)tile*TCOL + col];
      if (tb >= 0) {
        double *o = a.out + (size_t)(tb - a.box0)*a.nstored*PL;
        #pragma unroll
        for (int rb = 0; rb < NRB; ++rb)
          #pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int row = a.rowmap[16*rb + Mfma<T>::row(lane, i)];
            if (row >= 0)
              for (int q = 0; q < PL; ++q) o[(size_t)row*PL + q] = (double)acc[q][rb][i];
          }
      }
    } else {
      // slot 1: the block begins in this workgroup, slot 0: it began before
      T *o = static_cast<T *>(a.partial) +
             ((size_t)(2*g + (s0 == 0))*WAVES + wave)*(PL*NRB*256) + lane;
      #pragma unroll
      for (int q = 0; q < PL; ++q)
        #pragma unroll
        for (int rb = 0; rb < NRB; ++rb)
          #pragma unroll
          for (int i = 0; i < 4; ++i) o[((q*NRB + rb)*4 + i)*64] = acc[q][rb][i];
    }
  }
}

// out rows of the blocks whose slots lie in several workgroups: the sum in FP64
// of their partial accumulators in workgroup order
template <typename T, bool CX>
__global__ __launch_bounds__(256) void fold_reduce_kernel(ApplyArgs a, int nrb) {
  constexpr int PL = CX ? 2 : 1;
  const int b = blockIdx.x/WAVES, wave = blockIdx.x % WAVES;
  const int nsl = a.type_end[8*b + 7];
  if (nsl == 0) return;
  const long long cost = a.block_cost[a.nblocks], G = num_wg(a, cost);
  const long long g0 = wg_of(cost, a.block_cost[b], G);
  const long long g1 = wg_of(cost, a.block_cost[b] + a.slot_cost[(size_t)b*a.maxslots + nsl - 1], G);
  if (g0 == g1) return;
  const int lane = threadIdx.x & 63, i = threadIdx.x >> 6;
  const int tb = a.tile_target[((size_t)b*WAVES + wave)*TCOL + (lane & 15)];
  if (tb < 0) return;
  const size_t tile = (size_t)PL*nrb*256;
  const T *part = static_cast<const T *>(a.partial);
  for (int rb = blockIdx.y; rb < nrb; rb += gridDim.y) {
    const int row = a.rowmap[16*rb + Mfma<T>::row(lane, i)];
    if (row < 0) continue;
    for (int q = 0; q < PL; ++q) {
      const size_t e = ((size_t)q*nrb + rb)*256 + i*64 + lane;
      double s = part[((size_t)(2*g0 + 1)*WAVES + wave)*tile + e];
      for (long long g = g0 + 1; g <= g1; ++g) s += part[((size_t)(2*g)*WAVES + wave)*tile + e];
      a.out[((size_t)(tb - a.box0)*a.nstored + row)*PL + q] = s;
    }
  }
}

template <typename T, int ORD, bool CX>
constexpr size_t lds_bytes() {
  return 2*(CX ? 2 : 1)*Layout<ORD, sizeof(T) == 8>::SIZE*sizeof(T) + Fold<ORD>::NKP*4*sizeof(int2);
}

// raises the kernel's LDS limit where it needs more than 64 KiB
template <typename T, int ORD, bool CX>
int set_lds() {
  constexpr size_t bytes = lds_bytes<T, ORD, CX>();
  static_assert(bytes <= 160*1024, "class data exceed LDS");
  if (bytes <= 64*1024) return SUMPYHIP_OK;
  hipError_t e = hipFuncSetAttribute((const void *)fold_apply_kernel<T, ORD, CX>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e != hipSuccess)
    return set_error(SUMPYHIP_EHIP, "m2l_fold: cannot raise LDS limit to %zu: %s", bytes,
                     hipGetErrorString(e));
  return SUMPYHIP_OK;
}

template <typename T, int ORD, bool CX>
int launch_apply(const ApplyArgs &a, hipStream_t st) {
  int rc = set_lds<T, ORD, CX>();
  if (rc) return rc;
  fold_apply_kernel<T, ORD, CX><<<8*((a.max_wg + 7)/8), 256, lds_bytes<T, ORD, CX>(), st>>>(a);
  rc = check_launch("m2l_fold_apply");
  if (rc) return rc;
  constexpr int NRB = Fold<ORD>::NRB;
  fold_reduce_kernel<T, CX><<<dim3(a.nblocks*WAVES, NRB), 256, 0, st>>>(a, NRB);
  return check_launch("m2l_fold_reduce");
}

// workgroups of the contraction that the GPU holds at once
template <typename T, int ORD, bool CX>
int max_wg(int *out) {
  int per_cu = 0;
  int rc = set_lds<T, ORD, CX>();
  if (rc) return rc;
  hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(
      &per_cu, (const void *)fold_apply_kernel<T, ORD, CX>, 256, lds_bytes<T, ORD, CX>());
  if (e != hipSuccess)
    return set_error(SUMPYHIP_EHIP, "m2l_fold: occupancy: %s", hipGetErrorString(e));
  *out = num_cus()*(per_cu > 0 ? per_cu : 1);
  return SUMPYHIP_OK;
}

// the kernels of orders ORD..HI
template <typename T, bool CX, int ORD, int HI>
int dispatch_max_wg(int order, int *out) {
  if (order == ORD) return max_wg<T, ORD, CX>(out);
  if constexpr (ORD < HI) return dispatch_max_wg<T, CX, ORD + 1, HI>(order, out);
  return set_error(SUMPYHIP_ENOTIMPL, "m2l_fold: order %d (1..12)", order);
}

template <typename T, bool CX, int ORD, int HI>
int dispatch_apply(int order, const ApplyArgs &a, hipStream_t st) {
  if (order == ORD) return launch_apply<T, ORD, CX>(a, st);
  if constexpr (ORD < HI) return dispatch_apply<T, CX, ORD + 1, HI>(order, a, st);
  return set_error(SUMPYHIP_ENOTIMPL, "m2l_fold_apply: order %d (1..12)", order);
}

// }}}

// The kernels of orders LO..HI, a source file each: they compile side by side.
#define SUMPYHIP_FOLD_INSTANCE(NAME, T, CX, LO, HI)                                      \
  int m2l_fold_apply_##NAME(int order, const ApplyArgs &a, hipStream_t st) {             \
    return dispatch_apply<T, CX, LO, HI>(order, a, st);                                  \
  }                                                                                      \
  int m2l_fold_max_wg_##NAME(int order, int *out) {                                      \
    return dispatch_max_wg<T, CX, LO, HI>(order, out);                                   \
  }

}  // namespace m2l_fold
}  // namespace sumpyhip
