// FP64 stage kernel on v_mfma_f64_4x4x4_4b (stage-kernel variant 9).
//
// One wave owns a group of 8 elements and holds it as 16 columns: column
// 2 el + fld is field fld (0 = E, 1 = H) of element el. In the layout of
// v_mfma_f64_4x4x4_4b lane l = 16 q + c has column c of row q of B and of the
// result, so
//  * volume: the Np nodes are dealt into groups of four, node(g, q); lane q
//    of a column reads its three field components at node(b, q) from LDS and
//    they are the B operands of block column b as they stand. The product for
//    output group a, derivative k hands lane q the reference derivative at its
//    own node(a, q): J^-1, the curl and the accumulators never leave the lane;
//    the curl of one field is the other field's right-hand side and moves to
//    the neighbouring lane (l ^ 1) with a DPP quad permute.
//  * flux: lane q of a column owns local face q: one face code, one normal
//    and the face's Nfp nodes one after the other. The three flux components
//    of face node s are the B operands of LIFT's columns {f Nfp + s}, again as
//    they stand; the partner field's jump comes over the same DPP permute.
//    Neighbour nodes come from the face code and a 16-byte row of packed node
//    numbers in LDS (no per-face-node table is read from HBM).
//  * D_k is sparse on equispaced nodes: 4x4 blocks of D_k that are zero are
//    left out at compile time, and the node groups below are the ones an
//    annealed search found to leave the fewest: 20 of 27, 49 of 75 and 138 of
//    243 blocks at N = 2, 3, 4 (26 % to 43 % of the volume products).
//  * state in and stage update out are linear over the group (16-byte or
//    8 + 4 byte loads and stores per lane, no lane idle): y goes to LDS as FP64,
//    and the right-hand side comes back through the same LDS.
// On MI355X v_mfma_f64_4x4x4_4b runs at the vector unit's FP64 rate (70
// TFLOP/s measured, v_mfma_f64_16x16x4 48) and shares its cycles with vector
// instructions, so what it saves over FMAs is operand traffic (D and LIFT as
// one LDS read per 4 x 4 x 16 products instead of one per lane and node) and
// idle lanes (29 of 64 with one lane per node at N = 4).
//
// Compressed registers (CIN) take their sums in node order, by QuadRows: more
// blocks, the face fluxes formed per node as the one-lane-per-node kernels form
// them and moved between the lanes (transpose_rows), for the same bits.
//
// What bounds it (LSERK4 stage, FP64 registers, 324,000 tets at N = 3, 290 us
// against 416 for the variant before it): the memory side. Leaving out all
// products changes nothing, streaming the state and p alone takes 245 us (5.3
// TB/s), the neighbour traces, 10 M line requests to L2, the rest. At N = 4
// (384,000 tets, 690 us against 1232) products and vector instructions fill 47
// and 20 % of the issue cycles. Compressed registers: 262 us against 376 and 735
// against 1170, bound the same way (49 and 28 %).
#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "rfhip_elem_tables.hpp"
#include "rfhip_impl.hpp"
#include "rfhip_regs.hpp"

namespace rfhip {
namespace {

constexpr int kQuadEl = 8;  // elements per wave

// Node groups: NODE[g][q] is the node of lane q in group g (Np: none). NWB:
// waves per block (they share the tables in LDS). TW: neighbour traces
// requested ahead of the previous group's stores. RING: fragment pairs in
// registers. LATE: the state is read at the group's start and the update's
// registers after LIFT instead of one phase earlier, for want of registers: at
// N = 4 the early reads spill 34 to 100 of them, and since a reload waits in
// order behind the stores that costs more (929 us against 703 per FP64 stage
// of 384,000 tets). TW and RING are the fastest of 2 to 10 and 2 to 5.
template <int NP>
struct QuadTab;
template <>
struct QuadTab<4> {
  static constexpr int NG = 1, NWB = 4, TW = 3, RING = 4;
  static constexpr bool LATE = false;
  static constexpr int NODE[NG][4] = {{0, 1, 2, 3}};
};
template <>
struct QuadTab<10> {
  static constexpr int NG = 3, NWB = 4, TW = 6, RING = 4;
  static constexpr bool LATE = false;
  static constexpr int NODE[NG][4] = {{4, 1, 7, 2}, {10, 10, 9, 8}, {3, 6, 0, 5}};
};
template <>
struct QuadTab<20> {
  static constexpr int NG = 5, NWB = 4, TW = 4, RING = 4;
  static constexpr bool LATE = false;
  static constexpr int NODE[NG][4] = {{6, 3, 12, 2}, {17, 18, 19, 16}, {5, 0, 4, 1}, {14, 11, 10, 13}, {15, 9, 8, 7}};
};
template <>
struct QuadTab<35> {
  static constexpr int NG = 9, NWB = 8, TW = 2, RING = 3;
  static constexpr bool LATE = true;
  static constexpr int NODE[NG][4] = {{7, 11, 21, 8},  {30, 33, 28, 29}, {19, 20, 23, 22}, {9, 6, 10, 5}, {16, 15, 0, 1},
                                      {24, 12, 13, 14}, {4, 17, 3, 2},   {25, 18, 26, 27}, {32, 35, 31, 34}};
};

// The rows and columns of the products. SEQ: every sum takes its terms in
// node (and face node) order, as the one-lane-per-node kernels do, entries of
// D_k that are round-off residues included, so that with v_mfma_f64_4x4x4_4b's
// chain of FMAs in row order 0..3 the results are theirs bit for bit: the
// columns are dealt out in order, only the rows into the groups that leave the
// fewest blocks with entries that are not 0.0 (21 of 27, 66 of 75, 218 of 243).
template <int NP>
struct QuadRows;
template <>
struct QuadRows<4> {
  static constexpr int NODE[1][4] = {{0, 1, 2, 3}};
};
template <>
struct QuadRows<10> {
  static constexpr int NODE[3][4] = {{10, 2, 1, 0}, {5, 10, 3, 4}, {6, 9, 7, 8}};
};
template <>
struct QuadRows<20> {
  static constexpr int NODE[5][4] = {{16, 19, 10, 17}, {18, 13, 14, 7}, {8, 9, 5, 4}, {3, 0, 2, 1}, {6, 11, 12, 15}};
};
template <>
struct QuadRows<35> {
  static constexpr int NODE[9][4] = {{4, 1, 2, 3},     {19, 20, 22, 33}, {5, 14, 12, 9}, {27, 26, 17, 16}, {6, 13, 11, 10},
                                     {32, 25, 18, 15}, {31, 0, 34, 35},  {23, 28, 21, 8}, {30, 7, 24, 29}};
};
template <int NP, bool SEQ>
constexpr int quad_row(int a, int i) {
  return SEQ ? QuadRows<NP>::NODE[a][i] : QuadTab<NP>::NODE[a][i];
}
template <int NP, bool SEQ>
constexpr int quad_col(int b, int j) {
  return SEQ ? (4 * b + j < NP ? 4 * b + j : NP) : QuadTab<NP>::NODE[b][j];
}

// Whether block (a, b) of D_k has a nonzero.
template <int NP, bool SEQ>
constexpr bool quad_nz(int k, int a, int b) {
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 4; ++j) {
      const int r = quad_row<NP, SEQ>(a, i), c = quad_col<NP, SEQ>(b, j);
      if (r < NP && c < NP && (((SEQ ? ElemTab<NP>::XM : ElemTab<NP>::DM)[k][r] >> c) & 1ull)) return true;
    }
  return false;
}
// Blocks before (a, b, k) in the order the kernel reads them (k fastest);
// quad_at(NG, 0, 0) counts them all and LIFT's fragments start there.
template <int NP, bool SEQ>
constexpr int quad_at(int a_end, int b_end, int k_end) {
  int s = 0;
  for (int a = 0; a < QuadTab<NP>::NG; ++a)
    for (int b = 0; b < QuadTab<NP>::NG; ++b)
      for (int k = 0; k < 3; ++k) {
        if (a > a_end || (a == a_end && (b > b_end || (b == b_end && k >= k_end)))) return s;
        s += quad_nz<NP, SEQ>(k, a, b) ? 1 : 0;
      }
  return s;
}
// Steps of the volume: the blocks (a, b), a-major, where any D_k has a nonzero.
template <int NP, bool SEQ>
constexpr int quad_steps() {
  int n = 0;
  for (int ab = 0; ab < QuadTab<NP>::NG * QuadTab<NP>::NG; ++ab)
    n += quad_nz<NP, SEQ>(0, ab / QuadTab<NP>::NG, ab % QuadTab<NP>::NG) || quad_nz<NP, SEQ>(1, ab / QuadTab<NP>::NG, ab % QuadTab<NP>::NG) ||
         quad_nz<NP, SEQ>(2, ab / QuadTab<NP>::NG, ab % QuadTab<NP>::NG);
  return n;
}
template <int NP, bool SEQ>
constexpr int quad_step(int st) {
  constexpr int NG = QuadTab<NP>::NG;
  for (int ab = 0; ab < NG * NG; ++ab)
    if (quad_nz<NP, SEQ>(0, ab / NG, ab % NG) || quad_nz<NP, SEQ>(1, ab / NG, ab % NG) || quad_nz<NP, SEQ>(2, ab / NG, ab % NG))
      if (st-- == 0) return ab;
  return -1;
}
template <int NP, bool SEQ>
struct QuadSize {
  static constexpr int NV = quad_at<NP, SEQ>(QuadTab<NP>::NG, 0, 0);
  // LIFT's column steps: a node of every face, or (SEQ) four nodes of one face
  static constexpr int NU = (ElemTab<NP>::NFP + 3) / 4;
  static constexpr int NL = (SEQ ? 4 * NU : ElemTab<NP>::NFP) * QuadTab<NP>::NG;
  static constexpr int NF = NV + NL;  // A fragments of 16 doubles
};

template <int B, int E, class F>
__device__ __forceinline__ void unroll(F &&f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    unroll<B + 1, E>(f);
  }
}

// The value of the other field's lane of the same element (lane l ^ 1).
__device__ __forceinline__ double other_field(double v) {
  const int2 w = __builtin_bit_cast(int2, v);
  const int lo = __builtin_amdgcn_mov_dpp(w.x, 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(w.y, 0xB1, 0xF, 0xF, true);
  return __builtin_bit_cast(double, make_int2(lo, hi));
}

// The 4x4 transpose of four registers over the four rows of 16 lanes: row q of
// register f takes row f of register q.
__device__ __forceinline__ void transpose_rows(double &r0, double &r1, double &r2, double &r3) {
  uint2 v[4] = {__builtin_bit_cast(uint2, r0), __builtin_bit_cast(uint2, r1), __builtin_bit_cast(uint2, r2),
                __builtin_bit_cast(uint2, r3)};
  auto half = [](uint32_t &a, uint32_t &b) {  // rows 2, 3 of a with rows 0, 1 of b
    const auto t = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = t[0];
    b = t[1];
  };
  auto quarter = [](uint32_t &a, uint32_t &b) {  // rows 1, 3 of a with rows 0, 2 of b
    const auto t = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = t[0];
    b = t[1];
  };
  half(v[0].x, v[2].x);
  half(v[1].x, v[3].x);
  half(v[0].y, v[2].y);
  half(v[1].y, v[3].y);
  quarter(v[0].x, v[1].x);
  quarter(v[2].x, v[3].x);
  quarter(v[0].y, v[1].y);
  quarter(v[2].y, v[3].y);
  r0 = __builtin_bit_cast(double, v[0]);
  r1 = __builtin_bit_cast(double, v[1]);
  r2 = __builtin_bit_cast(double, v[2]);
  r3 = __builtin_bit_cast(double, v[3]);
}

// Two floats to bf16 (round to nearest even), a in the low half, as in
// rfhip_fused.hip (from (float)double operands the compiler rounds once).
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  const __bf16 x = (__bf16)a, y = (__bf16)b;
  return (uint32_t)__builtin_bit_cast(uint16_t, x) | ((uint32_t)__builtin_bit_cast(uint16_t, y) << 16);
}
__device__ __forceinline__ double c_f64(float h, uint32_t lo_bits) { return (double)h + (double)__uint_as_float(lo_bits); }

struct F3 {
  float x, y, z;
};
struct D3 {
  double x, y, z;
};
struct U2 {
  uint32_t x, y;
};

// Three values of one field at one node as stored: f32 + the 8 bytes that
// hold its bf16 parts, or f64.
template <bool CIN>
struct Trace;
template <>
struct Trace<true> {
  F3 h;
  U2 l;
};
template <>
struct Trace<false> {
  D3 d;
};

// VW consecutive values of a linear register as stored.
template <bool CIN, int VW>
struct Lin;
template <>
struct Lin<true, 4> {
  float4 h;
  uint2 l;
};
template <>
struct Lin<true, 2> {
  float2 h;
  uint32_t l;
};
template <int VW>
struct Lin<false, VW> {
  double2 d[VW / 2];
};

template <class T>
__device__ __forceinline__ T ld(const void *p, uint32_t byte) {
  T v;
  __builtin_memcpy(&v, static_cast<const char *>(p) + byte, sizeof(T));
  return v;
}
template <class T>
__device__ __forceinline__ T ld_al(const void *p, uint32_t byte) {
  return *reinterpret_cast<const T *>(static_cast<const char *>(p) + byte);
}
// Accesses of the update's registers and of every result, each touched once
// per launch. NT: streamed, kept from displacing the state that neighbours
// gather (quad_streams below says when).
template <bool NT, class T>
__device__ __forceinline__ T ld_reg(const void *p, uint32_t byte) {
  if constexpr (NT) {
    typedef unsigned W __attribute__((ext_vector_type(sizeof(T) / 4)));
    return __builtin_bit_cast(T, __builtin_nontemporal_load(reinterpret_cast<const W *>(static_cast<const char *>(p) + byte)));
  } else {
    return ld_al<T>(p, byte);
  }
}
template <bool NT, class T>
__device__ __forceinline__ void st_reg(void *p, uint32_t byte, T v) {
  if constexpr (NT) {
    typedef unsigned W __attribute__((ext_vector_type(sizeof(T) / 4)));
    __builtin_nontemporal_store(__builtin_bit_cast(W, v), reinterpret_cast<W *>(static_cast<char *>(p) + byte));
  } else {
    *reinterpret_cast<T *>(static_cast<char *>(p) + byte) = v;
  }
}

template <bool CIN, int VW, bool NT = false>
__device__ __forceinline__ Lin<CIN, VW> load_lin(const void *hi, const void *lo, uint32_t i) {
  auto get = [](auto z, const void *p, uint32_t byte) { return ld_reg<NT, decltype(z)>(p, byte); };
  Lin<CIN, VW> r;
  if constexpr (CIN && VW == 4) {
    r.h = get(float4{}, hi, 4 * i);
    r.l = get(uint2{}, lo, 2 * i);
  } else if constexpr (CIN) {
    r.h = get(float2{}, hi, 4 * i);
    r.l = get(uint32_t{}, lo, 2 * i);
  } else {
#pragma unroll
    for (int v = 0; v < VW / 2; ++v) r.d[v] = get(double2{}, hi, 8 * i + 16 * v);
  }
  return r;
}
template <bool CIN, int VW>
__device__ __forceinline__ void lin_f64(const Lin<CIN, VW> &r, double *v) {
  if constexpr (CIN && VW == 4) {
    v[0] = c_f64(r.h.x, r.l.x << 16);
    v[1] = c_f64(r.h.y, r.l.x & 0xFFFF0000u);
    v[2] = c_f64(r.h.z, r.l.y << 16);
    v[3] = c_f64(r.h.w, r.l.y & 0xFFFF0000u);
  } else if constexpr (CIN) {
    v[0] = c_f64(r.h.x, r.l << 16);
    v[1] = c_f64(r.h.y, r.l & 0xFFFF0000u);
  } else {
#pragma unroll
    for (int q = 0; q < VW / 2; ++q) {
      v[2 * q] = r.d[q].x;
      v[2 * q + 1] = r.d[q].y;
    }
  }
}
// VW FP64 values stored as f32 hi + bf16 lo.
template <bool NT, int VW>
__device__ __forceinline__ void store_c(void *hi, void *lo, uint32_t i, const double *v) {
  float h[VW], r[VW];
#pragma unroll
  for (int q = 0; q < VW; ++q) {
    h[q] = (float)v[q];
    r[q] = (float)(v[q] - (double)h[q]);
  }
  if constexpr (VW == 4) {
    st_reg<NT>(hi, 4 * i, make_float4(h[0], h[1], h[2], h[3]));
    st_reg<NT>(lo, 2 * i, make_uint2(bf16_pair(r[0], r[1]), bf16_pair(r[2], r[3])));
  } else {
    st_reg<NT>(hi, 4 * i, make_float2(h[0], h[1]));
    st_reg<NT>(lo, 2 * i, bf16_pair(r[0], r[1]));
  }
}
template <bool NT, int VW>
__device__ __forceinline__ void store_d(void *p, uint32_t i, const double *v) {
#pragma unroll
  for (int q = 0; q < VW / 2; ++q) st_reg<NT>(p, 8 * i + 16 * q, make_double2(v[2 * q], v[2 * q + 1]));
}
template <bool NT, int VW>
__device__ __forceinline__ void store_f(void *p, uint32_t i, const float *v) {
  if constexpr (VW == 4)
    st_reg<NT>(p, 4 * i, make_float4(v[0], v[1], v[2], v[3]));
  else
    st_reg<NT>(p, 4 * i, make_float2(v[0], v[1]));
}
template <int VW>
struct Flt {
  float v[VW];
};
template <bool NT, int VW>
__device__ __forceinline__ Flt<VW> load_f(const void *p, uint32_t i) {
  if constexpr (VW == 4) {
    const float4 t = ld_reg<NT, float4>(p, 4 * i);
    return {{t.x, t.y, t.z, t.w}};
  } else {
    const float2 t = ld_reg<NT, float2>(p, 4 * i);
    return {{t.x, t.y}};
  }
}

// The linear registers an epilogue reads besides the state: p (LSERK4) or y
// and err (KCL).
template <int EPI, int VW, bool NT>
struct Upd {};
template <int VW, bool NT>
struct Upd<1, VW, NT> {
  Lin<false, VW> p;
  __device__ __forceinline__ void load(const StageArgs &io, uint32_t i) { p = load_lin<false, VW, NT>(io.p, nullptr, i); }
};
template <int VW, bool NT>
struct Upd<2, VW, NT> {
  Flt<VW> p;
  __device__ __forceinline__ void load(const StageArgs &io, uint32_t i) { p = load_f<NT, VW>(io.p, i); }
};
template <int VW, bool NT>
struct Upd<3, VW, NT> {
  Lin<true, VW> y;
  Flt<VW> e;
  __device__ __forceinline__ void load(const StageArgs &io, uint32_t i) {
    y = load_lin<true, VW, NT>(io.ky, io.ky_lo, i);
    e = load_f<NT, VW>(io.kerr, i);
  }
};
template <int VW, bool NT>
struct Upd<4, VW, NT> {
  Lin<false, VW> y, e;
  __device__ __forceinline__ void load(const StageArgs &io, uint32_t i) {
    y = load_lin<false, VW, NT>(io.kyd, nullptr, i);
    e = load_lin<false, VW, NT>(io.kerrd, nullptr, i);
  }
};

__device__ __forceinline__ int64_t quad_block() {
  const unsigned nb = gridDim.x;
  return (nb & 7u) == 0 ? (int64_t)(blockIdx.x & 7u) * (nb >> 3) + (blockIdx.x >> 3) : (int64_t)blockIdx.x;
}

// Waves per SIMD the registers are fitted to: the most that leave no spills
// (N = 2: 300 us at 3 waves, 342 at 2 with compressed registers; 427 at 3 with
// 13 spilled, 350 at 2, with FP64 ones; N = 3 at 3 waves spills 48 to 100). At
// N = 1 the LSERK4 stage runs 4 waves fitted to 3 or to 4 (116 to 122 VGPRs),
// within 1 % of each other from 384 to 1.3M tets.
template <int NP, int EPI>
struct QuadWaves {
  static constexpr int v = NP == 4 ? (EPI <= 2 ? 4 : 3) : NP == 10 && (EPI == 0 || EPI == 2) ? 3 : 2;
};

// EPI as in the other stage kernels: 0 apply, 1 LSERK4 stage with FP64
// registers, 2 with compressed ones, 3 / 4 KCL stage with compressed / FP64
// registers. CIN: the input state is f32 + bf16. NT: quad_streams. nw: the
// waves of a block that take groups (all of them load the tables).
template <int NP, bool CIN, int EPI, bool NT>
__global__ void __launch_bounds__(QuadTab<NP>::NWB * 64) __attribute__((amdgpu_waves_per_eu(QuadWaves<NP, EPI>::v))) k_quad(StageArgs io, int nw) {
  using T = QuadTab<NP>;
  constexpr bool SEQ = CIN;
  using Z = QuadSize<NP, SEQ>;
  constexpr int NG = T::NG, NTH = T::NWB * 64, NFP = ElemTab<NP>::NFP;
  constexpr int SE = 6 * NP;             // values per element
  constexpr int SW = kQuadEl * SE;       // values per group
  // Element stride in LDS, = 4 mod 8 in 8-byte banks: with the nodes of lanes
  // q = 0, 1 (and 2, 3) of a group of different parity, the 32 lanes of a half
  // wave then read their 8-byte values from different banks.
  constexpr int SP = SE + (12 - SE % 8) % 8;
  constexpr int SZ = kQuadEl * SP;
  constexpr int VW = CIN && SE % 4 == 0 ? 4 : 2;
  constexpr int IT = (SW / VW + 63) / 64;
  constexpr int NFR = (Z::NF + 1) / 2;   // fragment pairs
  __shared__ __align__(16) double sA[NFR * 32];
  __shared__ __align__(16) uint4 snode[100];
  __shared__ int splace[2][4 * NG];  // LDS place in an element of column (0) and row (1) node (g, q)
  __shared__ __align__(16) double su_b[T::NWB][SZ + 8];  // + zeros the padding nodes read, + a place for what they write
  for (int t = threadIdx.x; t < NFR * 16; t += NTH) reinterpret_cast<double2 *>(sA)[t] = reinterpret_cast<const double2 *>(SEQ ? io.quad_seq : io.quad)[t];
  for (int t = threadIdx.x; t < 100; t += NTH) snode[t] = reinterpret_cast<const uint4 *>(io.quad_nodes)[t];
  if ((int)threadIdx.x < 4 * NG) {
    const int g = threadIdx.x >> 2, r = threadIdx.x & 3;
    splace[1][threadIdx.x] = 6 * quad_row<NP, SEQ>(g, r);
    splace[0][threadIdx.x] = 6 * quad_col<NP, SEQ>(g, r);
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  double *su = su_b[wave];
  double2 *su2 = reinterpret_cast<double2 *>(su);
  auto at = [](int i) { return i + (i / SE) * (SP - SE); };  // LDS place of value i of the group
  const int64_t ngroups = (io.n_elem + kQuadEl - 1) / kQuadEl;
  const int64_t gw0 = quad_block() * nw + wave, gws = (int64_t)gridDim.x * nw;
  __syncthreads();  // the only block-wide barrier: the tables are in LDS
  auto wave_sync = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  if (lane < 4) su[SZ + lane] = 0.0;
  const int64_t wslot = (int64_t)blockIdx.x * nw + wave;
  double wsum = 0.0;
  if (wave >= nw || gw0 >= ngroups) {
    if constexpr (EPI == 3 || EPI == 4)
      if (wave < nw && io.klast && (threadIdx.x & 63) == 0) io.kpart[wslot] = 0.0;
    return;
  }
  const int q = lane >> 4, fld = lane & 1, el = (lane >> 1) & 7;
  // A operand: lane 16 kk + 4 b + i reads entry (kk, i) of a fragment for every b; pair t: fr[16 t]
  const double2 *fr = reinterpret_cast<const double2 *>(sA) + (4 * q + (lane & 3));
  // LDS index of this lane's three values at node(g, q), from a table where
  // they are used (held for the whole group they would cost NG registers).
  auto places = [&](int (&un)[NG], int rc) {
    int t = q;
    asm volatile("" : "+v"(t));
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int n = splace[rc][4 * g + t];
      un[g] = n < SE ? el * SP + n + 3 * fld : SZ;
    }
  };

  // Every load a group needs before its LIFT is issued ahead of the stores of
  // the group before it: its state (nx), J^-1, materials and first neighbour
  // traces. Vector memory operations retire in order, so a load behind those
  // stores would be waited for together with them. Face codes and material
  // indices, which those loads depend on, run two groups ahead.
  // All loads are unconditional, with clamped indices.
  Lin<CIN, VW> nx[IT];
  auto read_state = [&](int64_t g, int ln) {
    const int64_t rg = io.n_elem - g * kQuadEl;
    const int ng = rg < kQuadEl ? (int)rg : kQuadEl;
    const uint32_t gb = (uint32_t)g * SW, last = gb + (uint32_t)(ng * SE - VW);
#pragma unroll
    for (int k = 0; k < IT; ++k) {
      const uint32_t i = gb + (uint32_t)(ln + 64 * k) * VW;
      nx[k] = load_lin<CIN, VW>(io.yin, io.yin_lo, i < last ? i : last);
    }
  };
  auto elem_of = [&](int64_t g) {
    const int64_t rg = io.n_elem - g * kQuadEl;
    const int ng = rg < kQuadEl ? (int)rg : kQuadEl;
    return (uint32_t)g * kQuadEl + (uint32_t)(el < ng ? el : ng - 1);
  };
  auto node_of = [](const uint4 &r, int s) {
    const uint32_t w = s < 4 ? r.x : s < 8 ? r.y : s < 12 ? r.z : r.w;
    return (w >> (8 * (s & 3))) & 0xFFu;
  };
  // A window of TW neighbour traces is in flight: each slot, once used, takes
  // the trace TW face nodes on. A wall or port face reads its own trace.
  constexpr int TW = NFP < T::TW ? NFP : T::TW;
  constexpr bool ROLL = T::LATE;
  constexpr int NTR = ROLL ? TW : NFP;
  Trace<CIN> tr[NTR];
  uint4 nrow;
  uint32_t tbh, tbl;
  auto load_trace = [&](int s) {
    const uint32_t n = node_of(nrow, s);
    if constexpr (CIN) {
      tr[s % NTR].h = ld<F3>(io.yin, tbh + 24 * n);
      tr[s % NTR].l = ld<U2>(io.yin_lo, tbl + 12 * n);
    } else {
      tr[s % NTR].d = ld<D3>(io.yin, tbh + 48 * n);
    }
  };
  struct J9 {
    double v[9];
  };
  J9 jr;
  auto read_geom = [&](int64_t g, int code) {
    const uint32_t e = elem_of(g);
    const int bnd = code >> 31;  // all ones on a wall or port face; masks, not a lane-divergent branch
    const uint32_t ne = (uint32_t)(((code >> 5) & ~bnd) | ((int)e & bnd));
    nrow = snode[((24 * q + 6 * ((code >> 3) & 3) + (code & 7)) & ~bnd) | ((96 + q) & bnd)];
    tbh = ne * (uint32_t)(SE * (CIN ? 4 : 8)) + (CIN ? 12 : 24) * fld;
    tbl = ne * (uint32_t)(2 * SE) + 4 * fld;
    jr = ld<J9>(io.jinv, 72 * e);
#pragma unroll
    for (int s = 0; s < TW; ++s) load_trace(s);
  };
  auto next_of = [&](int64_t g) { return g + gws < ngroups ? g + gws : g; };
  int code, mat, ncode, nmat;
  {
    const uint32_t e0 = elem_of(gw0), e1 = elem_of(next_of(gw0));
    code = io.fcode[4 * e0 + q];
    mat = io.mat[e0];
    ncode = io.fcode[4 * e1 + q];
    nmat = io.mat[e1];
    read_state(gw0, lane);
    read_geom(gw0, code);
  }

#pragma unroll 1
  for (int64_t grp = gw0; grp < ngroups; grp += gws) {
    const int64_t rem = io.n_elem - grp * kQuadEl;
    const int nel = rem < kQuadEl ? (int)rem : kQuadEl;
    const uint32_t gb = (uint32_t)grp * SW;
    // An opaque copy of the lane id, so the places of this lane's linear
    // values are formed where they are used and not held in registers.
    int ln = lane;
    asm volatile("" : "+v"(ln));

    if constexpr (T::LATE) read_state(grp, ln);
    // the group's state to LDS
#pragma unroll
    for (int k = 0; k < IT; ++k) {
      const int i = (ln + 64 * k) * VW;
      const int to = (SW / VW) % 64 == 0 || k < IT - 1 || i < SW ? at(i) : SZ + 4;
      double v[VW];
      lin_f64<CIN, VW>(nx[k], v);
#pragma unroll
      for (int c = 0; c < VW / 2; ++c) su2[to / 2 + c] = make_double2(v[2 * c], v[2 * c + 1]);
    }
    if constexpr (!ROLL) {
#pragma unroll
      for (int s = TW; s < NFP; ++s) load_trace(s);
    }
    double ji[9];
    {
      const double sg = fld ? 1.0 : -1.0;  // the curl of E enters dH/dt with a minus, and so does n x [H] dE/dt
#pragma unroll
      for (int c = 0; c < 9; ++c) ji[c] = sg * jr.v[c];
    }
    wave_sync();

    // Fragment pairs are read kRing - 1 pairs ahead of their products, in an
    // order the scheduler may not change: left to it, every read is issued
    // right before its first product and waited for there.
    constexpr int kRing = T::RING;
    double2 ring[kRing];
#pragma unroll
    for (int t = 0; t < kRing - 1; ++t) ring[t] = fr[16 * t];
    auto frag = [&](auto fc) {
      constexpr int t = fc / 2, ahead = t + kRing - 1;
      if constexpr (fc % 2 == 0) {
        if constexpr (ahead < NFR) ring[ahead % kRing] = fr[16 * ahead];
        if constexpr (fc < Z::NV) __builtin_amdgcn_sched_barrier(0);
      }
      return fc % 2 ? ring[t % kRing].y : ring[t % kRing].x;
    };

    // Volume: reference derivatives of this lane's field at its nodes, J^-1,
    // the curl, and over to the other field. The state operands come from LDS,
    // one block ahead of their products (held in registers for the whole
    // volume they would cost 6 Np / 4 of them).
    double acc[NG][3];
    double ub[2][3];
    int un[NG];
    places(un, 0);
    auto operand = [&](auto bc) {
      constexpr int st = bc;  // step: block (a, b) = (quad_step / NG, quad_step % NG)
      constexpr int ab = quad_step<NP, SEQ>(st);
#pragma unroll
      for (int c = 0; c < 3; ++c) ub[st & 1][c] = su[un[ab % NG] + c];
    };
    constexpr int NST = quad_steps<NP, SEQ>();
    operand(std::integral_constant<int, 0>{});
    double r[3][3];
    unroll<0, NST>([&](auto sc) {
      constexpr int st = sc, ab = quad_step<NP, SEQ>(st), a = ab / NG, b = ab % NG;
      if constexpr (st == 0 || quad_step<NP, SEQ>(st - 1) / NG != a) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
          for (int c = 0; c < 3; ++c) r[k][c] = 0.0;
      }
      if constexpr (st + 1 < NST) operand(std::integral_constant<int, st + 1>{});
      unroll<0, 3>([&](auto kc) {
        constexpr int k = kc;
        if constexpr (quad_nz<NP, SEQ>(k, a, b)) {
          const double f = frag(std::integral_constant<int, quad_at<NP, SEQ>(a, b, k)>{});
#pragma unroll
          for (int c = 0; c < 3; ++c) r[k][c] = __builtin_amdgcn_mfma_f64_4x4x4f64(f, ub[st & 1][c], r[k][c], 0, 0, 0);
        }
      });
      if constexpr (st + 1 == NST || quad_step<NP, SEQ>(st + 1) / NG != a) {
        auto pd = [&](int p, int c) {
          double t = fma(ji[p], r[0][c], ji[3 + p] * r[1][c]);
          // k_fused9 at Np = 35 starts E_x's two sums with the other product
          if (SEQ && NP == 35 && c == 0) t = fld ? t : fma(ji[3 + p], r[1][c], ji[p] * r[0][c]);
          return fma(ji[6 + p], r[2][c], t);
        };
        acc[a][0] = other_field(pd(1, 2) - pd(2, 1));
        acc[a][1] = other_field(pd(2, 0) - pd(0, 2));
        acc[a][2] = other_field(pd(0, 1) - pd(1, 0));
      }
    });

    // The next group's state and the registers the update reads, linear like
    // the state; requested here so the flux and LIFT cover their latency (the
    // volume's operands are free).
    __builtin_amdgcn_sched_barrier(0);
    const int64_t grp1 = next_of(grp);
    if constexpr (!T::LATE) read_state(grp1, ln);
    int nncode, nnmat;
    {
      const uint32_t e2 = elem_of(next_of(grp1));
      nncode = io.fcode[4 * e2 + q];
      nnmat = io.mat[e2];
    }
    constexpr bool kLateRegs = T::LATE || EPI == 4;
    Upd<EPI, VW, NT> up[EPI == 0 ? 1 : IT];
    auto read_registers = [&] {
      if constexpr (EPI != 0) {
        const uint32_t last = gb + (uint32_t)(nel * SE - VW);
#pragma unroll
        for (int k = 0; k < IT; ++k) {
          const uint32_t i = gb + (uint32_t)(ln + 64 * k) * VW;
          up[k].load(io, i < last ? i : last);
        }
      }
    };
    if constexpr (!kLateRegs) read_registers();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");

    D3 minv, msig;
    auto read_materials = [&] {
      minv = ld<D3>(io.mat_tab, 96 * (uint32_t)mat + 24 * fld);
      msig = ld<D3>(io.mat_tab, 96 * (uint32_t)mat + 48 + 24 * fld);
    };
    const double *const us = su + el * SP + 3 * fld;
    int qo = 96 + q;
    asm volatile("" : "+v"(qo));  // not a loop constant held in registers
    const uint4 orow = snode[qo];
    double ow[3];
    auto own_trace = [&](int s) {
      const double *p = us + node_of(orow, s) * 6;
      ow[0] = p[0];
      ow[1] = p[1];
      ow[2] = p[2];
    };
    // The jump j = own + sx * neighbour of slot s in this lane's field. On a
    // boundary face the trace read is the own one, and since the flux keeps
    // the tangential part of either jump, the wall and port rules are this
    // sign: PEC j = E (doubled in the flux) and 0, port j = own.
    auto jump = [&](auto sc, double sx, double (&j)[3]) {
      constexpr int s = sc;
      const Trace<CIN> x = tr[s % NTR];
      if constexpr (CIN) {
        const uint32_t sh = fld << 4;
        const uint32_t l0 = __builtin_amdgcn_alignbit(x.l.y, x.l.x, sh), l1 = x.l.y >> sh;
        j[0] = fma(sx, c_f64(x.h.x, l0 << 16), ow[0]);
        j[1] = fma(sx, c_f64(x.h.y, l0 & 0xFFFF0000u), ow[1]);
        j[2] = fma(sx, c_f64(x.h.z, l1 << 16), ow[2]);
      } else {
        j[0] = fma(sx, x.d.x, ow[0]);
        j[1] = fma(sx, x.d.y, ow[1]);
        j[2] = fma(sx, x.d.z, ow[2]);
      }
      if constexpr (ROLL && s + TW < NFP) load_trace(s + TW);
      if constexpr (s + 1 < NFP) own_trace(s + 1);
    };
    // Weights 0, +-1 per lane that make face q's vector of J^-1's rows without
    // branches; the sums of the other rows' zeros are exact.
    const double wr0 = q == 1 ? -1.0 : q == 3 ? 1.0 : 0.0, wr1 = q == 2 ? -1.0 : q == 3 ? 1.0 : 0.0,
                 wr2 = q == 0 ? -1.0 : q == 3 ? 1.0 : 0.0;
    if constexpr (SEQ) {
      // The operations and their order are face_geom's and face_flux's. n has
      // this lane's sign (E: -n), which the products n (n.j) do not see.
      double g[3];
#pragma unroll
      for (int x = 0; x < 3; ++x) g[x] = fma(wr2, ji[6 + x], fma(wr0, ji[x], wr1 * ji[3 + x]));
      const double gs = fma(g[2], g[2], fma(g[0], g[0], g[1] * g[1])), hs = 0.5 * gs;
      double iy = __builtin_amdgcn_rsq(gs);
      iy = iy * fma(-hs * iy, iy, 1.5);
      iy = iy * fma(-hs * iy, iy, 1.5);
      const double n0 = g[0] * iy, n1 = g[1] * iy, n2 = g[2] * iy;
      const bool pec = code == kCodePec;
      const double cf = (pec ? (fld ? 2.0 : 2.0 * io.alpha) : 1.0) * (hs * iy);
      const double al = code < 0 ? 1.0 : io.alpha;
      const double sx = code >= 0 ? -1.0 : pec && fld ? -1.0 : 0.0;
      double F[4 * Z::NU][3];
      own_trace(0);
      unroll<0, 4 * Z::NU>([&](auto sc) {
        constexpr int s = sc;
        if constexpr (s < NFP) {
          double j[3], o[3];
          jump(sc, sx, j);
#pragma unroll
          for (int c = 0; c < 3; ++c) o[c] = other_field(j[c]);
          const double nj = fma(n2, j[2], fma(n0, j[0], n1 * j[1]));
          F[s][0] = cf * fma(al, fma(n0, nj, -j[0]), fma(n1, o[2], -(n2 * o[1])));
          F[s][1] = cf * fma(al, fma(n1, nj, -j[1]), fma(n2, o[0], -(n0 * o[2])));
          F[s][2] = cf * fma(al, fma(n2, nj, -j[2]), fma(n0, o[1], -(n1 * o[0])));
        } else {
          F[s][0] = F[s][1] = F[s][2] = 0.0;
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      // Four nodes of four faces: from (node, lane = face) to (face, lane = node).
#pragma unroll
      for (int u = 0; u < Z::NU; ++u)
#pragma unroll
        for (int c = 0; c < 3; ++c) transpose_rows(F[4 * u][c], F[4 * u + 1][c], F[4 * u + 2][c], F[4 * u + 3][c]);
      unroll<0, 4>([&](auto fc) {
        unroll<0, Z::NU>([&](auto uc) {
          constexpr int f = fc, u = uc;
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (f == 3 && u == 0) read_materials();
          unroll<0, NG>([&](auto ac) {
            constexpr int a = ac;
            const double w = frag(std::integral_constant<int, Z::NV + (f * Z::NU + u) * NG + a>{});
#pragma unroll
            for (int c = 0; c < 3; ++c)
              acc[a][c] = __builtin_amdgcn_mfma_f64_4x4x4f64(w, F[4 * u + f][c], acc[a][c], 0, 0, 0);
          });
        });
      });
    } else {
      // m = -+ 0.5 g = -+ cf n of face q (sign as ji), cf = |m|.
      double m[3];
#pragma unroll
      for (int x = 0; x < 3; ++x) m[x] = 0.5 * (wr0 * ji[x] + wr1 * ji[3 + x] + wr2 * ji[6 + x]);
      const double ss = m[0] * m[0] + m[1] * m[1] + m[2] * m[2], hs = 0.5 * ss;
      double ic = __builtin_amdgcn_rsq(ss);  // 1 / cf, two Newton steps as in face_geom
      ic = ic * fma(-hs * ic, ic, 1.5);
      ic = ic * fma(-hs * ic, ic, 1.5);
      const double al = code < kCodePec ? 1.0 : io.alpha;
      const double acf = al * (ss * ic), aic = al * ic;
      // Flux and LIFT, one face node of every face at a time:
      // F = m (m . j) a / cf - a cf j -+ m x j' (j: this field's jump, j' the
      // other's; PEC j = 2 E and 0). The flux of a node is formed while the
      // products of the node before it run.
      const double sx = code >= 0 ? -1.0 : code < kCodePec ? 0.0 : fld ? -1.0 : 1.0;
      double F[2][3];
      own_trace(0);
      auto flux = [&](auto sc) {
        constexpr int s = sc;
        double j[3], o[3];
        jump(sc, sx, j);
#pragma unroll
        for (int c = 0; c < 3; ++c) o[c] = other_field(j[c]);
        const double t = aic * (m[0] * j[0] + m[1] * j[1] + m[2] * j[2]);
        F[s & 1][0] = m[0] * t - acf * j[0] + (m[1] * o[2] - m[2] * o[1]);
        F[s & 1][1] = m[1] * t - acf * j[1] + (m[2] * o[0] - m[0] * o[2]);
        F[s & 1][2] = m[2] * t - acf * j[2] + (m[0] * o[1] - m[1] * o[0]);
      };
      flux(std::integral_constant<int, 0>{});
      unroll<0, NFP>([&](auto sc) {
        constexpr int s = sc;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (s == (NFP > 3 ? NFP - 3 : 0)) read_materials();
        if constexpr (s + 1 < NFP) flux(std::integral_constant<int, s + 1>{});
        unroll<0, NG>([&](auto ac) {
          constexpr int a = ac;
          const double f = frag(std::integral_constant<int, Z::NV + s * NG + a>{});
#pragma unroll
          for (int c = 0; c < 3; ++c) acc[a][c] = __builtin_amdgcn_mfma_f64_4x4x4f64(f, F[s & 1][c], acc[a][c], 0, 0, 0);
        });
      });
    }

    // Materials (rhs.rs:1443-1454), then the right-hand side to LDS in place
    // of the state, which the update takes into registers first.
    auto rhs = [](double mi, double a, double ms, double u) {
      if constexpr (SEQ)
        return fma(mi, a, -(ms * u));
      else
        return mi * a - ms * u;
    };
    int up_at[NG];
    places(up_at, 1);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      acc[g][0] = rhs(minv.x, acc[g][0], msig.x, su[up_at[g]]);
      acc[g][1] = rhs(minv.y, acc[g][1], msig.y, su[up_at[g] + 1]);
      acc[g][2] = rhs(minv.z, acc[g][2], msig.z, su[up_at[g] + 2]);
    }
    // the next group's geometry and traces, ahead of this group's stores
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kLateRegs) read_registers();
    code = ncode;
    mat = nmat;
    read_geom(grp1, code);
    ncode = nncode;
    nmat = nnmat;
    __builtin_amdgcn_sched_barrier(0);
    double yv[EPI == 1 || EPI == 2 ? IT : 1][VW];
    if constexpr (EPI == 1 || EPI == 2) {
#pragma unroll
      for (int k = 0; k < IT; ++k) {
        const int i = (ln + 64 * k) * VW, ic2 = i < SW ? i : 0;
#pragma unroll
        for (int c = 0; c < VW / 2; ++c) {
          const double2 t = su2[at(ic2) / 2 + c];
          yv[k][2 * c] = t.x;
          yv[k][2 * c + 1] = t.y;
        }
      }
    }
    wave_sync();
    unroll<0, NG>([&](auto gc) {
      constexpr int g = gc;
      constexpr bool pad = quad_row<NP, SEQ>(g, 0) >= NP || quad_row<NP, SEQ>(g, 1) >= NP ||
                           quad_row<NP, SEQ>(g, 2) >= NP || quad_row<NP, SEQ>(g, 3) >= NP;
      const int to = pad && up_at[g] >= SZ ? SZ + 4 : up_at[g];
#pragma unroll
      for (int c = 0; c < 3; ++c) su[to + c] = acc[g][c];
    });
    wave_sync();
    const int nv = nel * SE;
    auto update = [&](auto full) {
      constexpr int CH = T::LATE ? 2 : 4;  // iterations of right-hand sides in registers at a time
#pragma unroll
      for (int k0 = 0; k0 < IT; k0 += CH) {
        double kr[CH][VW];
#pragma unroll
        for (int k = k0; k < (k0 + CH < IT ? k0 + CH : IT); ++k) {
          const int i = (ln + 64 * k) * VW, ic2 = i < SW ? i : 0;
#pragma unroll
          for (int c = 0; c < VW / 2; ++c) {
            const double2 t = su2[at(ic2) / 2 + c];
            kr[k - k0][2 * c] = t.x;
            kr[k - k0][2 * c + 1] = t.y;
          }
        }
        if (io.src_kind == RFHIP_DRIVE_POINT) {
          const int64_t off = io.src_dof - (int64_t)gb;
#pragma unroll
          for (int k = k0; k < (k0 + CH < IT ? k0 + CH : IT); ++k)
#pragma unroll
            for (int c = 0; c < VW; ++c)
              if (off == (ln + 64 * k) * VW + c) kr[k - k0][c] += io.g;
        } else if (io.src_kind == RFHIP_DRIVE_VECTOR) {
#pragma unroll
          for (int k = k0; k < (k0 + CH < IT ? k0 + CH : IT); ++k) {
            const int i = (ln + 64 * k) * VW;
            const double *sv = io.src_vec + gb + (i < nv ? i : 0);
#pragma unroll
            for (int c = 0; c < VW; ++c) kr[k - k0][c] += sv[c] * io.g;
          }
        }
#pragma unroll
        for (int k = k0; k < (k0 + CH < IT ? k0 + CH : IT); ++k) {
          const int i = (ln + 64 * k) * VW;
          if ((full && ((SW / VW) % 64 == 0 || k < IT - 1)) || i < nv) {
            const double *kv = kr[k - k0];
            const uint32_t gi = gb + (uint32_t)i;
            if constexpr (EPI == 0) {
              store_d<NT, VW>(io.dy, gi, kv);
            } else if constexpr (EPI == 1) {
              double po[VW], pn[VW], yn[VW];
              lin_f64<false, VW>(up[k].p, po);
    #pragma unroll
              for (int c = 0; c < VW; ++c) {
                pn[c] = io.sa * po[c] + io.dt * kv[c];
                yn[c] = yv[k][c] + io.sb * pn[c];
              }
              store_d<NT, VW>(io.p, gi, pn);
              store_d<NT, VW>(io.yout, gi, yn);
            } else if constexpr (EPI == 2) {
              float pn[VW];
              double yn[VW];
    #pragma unroll
              for (int c = 0; c < VW; ++c) {
                // which product is rounded on its own: dt k in E_x (i = 0 mod 6), a p in the rest
                const double po = up[k].p.v[c];
                double v = fma(io.dt, kv[c], io.sa * po);
                if (c % 2 == 0) v = (i + c) % 6 == 0 ? fma(io.sa, po, io.dt * kv[c]) : v;
                pn[c] = (float)v;
                yn[c] = fma(io.sb, (double)pn[c], yv[k][c]);
              }
              store_f<NT, VW>(io.p, gi, pn);
              store_c<NT, VW>(io.yout, io.yout_lo, gi, yn);
            } else if constexpr (EPI == 3) {
              // the arithmetic of node_kcl (rfhip_fused.hip)
              float en[VW];
              double yn[VW], sn[VW], yo[VW], bo[VW];
              if (io.klast) lin_f64<true, VW>(load_lin<true, VW>(io.kbak, io.kbak_lo, gi), bo);
              lin_f64<true, VW>(up[k].y, yo);
    #pragma unroll
              for (int c = 0; c < VW; ++c) {
                const double f = io.dt * kv[c];
                yn[c] = yo[c] + io.kb * f;
                const double er = io.kfirst ? io.kew * f : (double)up[k].e.v[c] + io.kew * f;
                en[c] = (float)er;
                sn[c] = io.klast ? yn[c] : yn[c] + io.kamb * f;
                if (io.klast) wsum += werr_term(bo[c], yn[c], er, io.katol, io.krtol);
              }
              store_c<NT, VW>(io.ky, io.ky_lo, gi, yn);
              store_f<NT, VW>(io.kerr, gi, en);
              store_c<NT, VW>(io.yout, io.yout_lo, gi, sn);
              if (io.kfirst) {
                st_reg<NT>(io.kbak, 4 * gi, up[k].y.h);
                st_reg<NT>(io.kbak_lo, 2 * gi, up[k].y.l);
              }
            } else {
              // the arithmetic of node_kcl64
              double yo[VW], er[VW], bo[VW], sn[VW], yn[VW];
              lin_f64<false, VW>(up[k].y, yo);
              lin_f64<false, VW>(up[k].e, er);
              if (io.klast) lin_f64<false, VW>(load_lin<false, VW>(io.kbakd, nullptr, gi), bo);
    #pragma unroll
              for (int c = 0; c < VW; ++c) {
                const double f = io.dt * kv[c];
                yn[c] = yo[c] + io.kb * f;
                er[c] = io.kfirst ? io.kew * f : er[c] + io.kew * f;
                sn[c] = io.klast ? yn[c] : yn[c] + io.kamb * f;
                if (io.klast) wsum += werr_term(bo[c], yn[c], er[c], io.katol, io.krtol);
              }
              store_d<NT, VW>(io.kyd, gi, yn);
              store_d<NT, VW>(io.kerrd, gi, er);
              store_d<NT, VW>(io.yout, gi, sn);
              if (io.kfirst) store_d<NT, VW>(io.kbakd, gi, yo);
            }
          }
        }
      }
    };
    if (nel == kQuadEl)
      update(std::true_type{});
    else
      update(std::false_type{});
    wave_sync();  // su takes the next group's state
  }
  if constexpr (EPI == 3 || EPI == 4) {
    if (io.klast) {
      // fixed butterfly order: the same sum for the same grid
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) wsum += __shfl_xor(wsum, o, 64);
      if ((threadIdx.x & 63) == 0) io.kpart[wslot] = wsum;
    }
  }
}

// Compute units of the current device and the blocks of `kernel` (nt threads)
// resident on one, looked up once per (kernel, device).
struct Residency {
  int64_t cus, per_cu;
};
inline Residency quad_resident(const void *kernel, int nt) {
  int dev = 0;
  RF_HIP(hipGetDevice(&dev));
  static std::mutex mu;
  static std::map<std::tuple<const void *, int>, Residency> cache;
  const auto key = std::make_tuple(kernel, dev);
  {
    std::lock_guard<std::mutex> lock(mu);
    const auto it = cache.find(key);
    if (it != cache.end()) return it->second;
  }
  int cus = 0, per_cu = 0;
  RF_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  RF_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, nt, 0));
  const Residency r{cus > 0 ? cus : 1, per_cu > 0 ? per_cu : 1};
  std::lock_guard<std::mutex> lock(mu);
  cache.emplace(key, r);
  return r;
}

// Blocks and waves per block: the persistent grid, at most the resident
// blocks. A mesh with fewer groups than a block per compute unit would hold
// gives fewer waves of each block a group instead of launching fewer blocks,
// so that its waves do not share a unit while others idle.
struct QuadGrid {
  int64_t blocks;
  int waves;
};
template <int NP, bool CIN, int EPI, bool NT>
QuadGrid quad_grid(int64_t n_elem) {
  constexpr int NWB = QuadTab<NP>::NWB;
  const int64_t groups = (n_elem + kQuadEl - 1) / kQuadEl;
  const Residency r = quad_resident(reinterpret_cast<const void *>(&k_quad<NP, CIN, EPI, NT>), NWB * 64);
  const int64_t nw = std::min<int64_t>(NWB, std::max<int64_t>(1, (groups + r.cus - 1) / r.cus));
  return {std::min((groups + nw - 1) / nw, r.cus * r.per_cu), (int)nw};
}
// Bytes of one value in the registers that an epilogue's launches alternate
// between: state in and out and p, or state in and out, y, err and the backup.
constexpr int quad_value_bytes(int epi) { return epi == 1 ? 24 : epi == 2 ? 16 : epi == 3 ? 28 : 40; }

// Whether the registers are streamed. A step's launches return to the same
// registers, and where those of this operator (with its geometry, 92 bytes an
// element) and of what is stepped beside it fit the 256 MB last-level cache, a
// streamed store sends out of it what the next launch reads. us per stage,
// streamed / not, FP64 registers: N = 1, 196,608 tets (131 MB) 43.2 / 33.3 (the
// fastest other variant 41.9), N = 4, 48,000 tets (246 MB) 100 / 98; above that
// size what passes through should not displace the state: N = 1, 511,104 tets
// (341 MB) 106 / 116, N = 3, 196,608 tets (584 MB) 175 / 189. Small registers
// are faster streamed too: N = 1, 12,096 tets (8 MB) 6.3 / 6.9, N = 3, 6,000 tets
// (18 MB) 10.8 / 11.5, then N = 1, 36,936 tets (25 MB) 14.4 / 12.3; compressed
// ones 13.2 / 13.5 there (18 MB) and 22.8 / 22.1 at 101,400 tets (48 MB). The
// apply (EPI 0) always streams: nothing returns to its result (the same within
// 1 % up to 300 MB, 3 % faster above).
bool quad_streams(int np, bool cin, int epi, const StageArgs &a) {
  const int64_t mb = (int64_t)1 << 20;
  const int64_t own = a.n_elem * (6 * np * quad_value_bytes(epi) + 92);
  return epi == 0 || own < (cin ? 32 : 20) * mb || own + a.beside > 256 * mb;
}
template <int NP, bool CIN, int EPI, bool NT>
void quad_launch_nt(const StageArgs &a, hipStream_t s) {
  const QuadGrid g = quad_grid<NP, CIN, EPI, NT>(a.n_elem);
  if (g.blocks > 0) hipLaunchKernelGGL((k_quad<NP, CIN, EPI, NT>), dim3((unsigned)g.blocks), dim3(QuadTab<NP>::NWB * 64), 0,
                       s, a, g.waves);
}
template <int NP, bool CIN, int EPI>
void quad_launch(const StageArgs &a, hipStream_t s) {
  if (EPI == 0 || quad_streams(NP, CIN, EPI, a))
    quad_launch_nt<NP, CIN, EPI, true>(a, s);
  else
    quad_launch_nt<NP, CIN, EPI, EPI == 0>(a, s);
}
template <int NP, bool CIN, int EPI>
int64_t quad_slots_epi(const StageArgs &a) {
  const QuadGrid g = quad_streams(NP, CIN, EPI, a) ? quad_grid<NP, CIN, EPI, true>(a.n_elem)
                                                   : quad_grid<NP, CIN, EPI, false>(a.n_elem);
  return g.blocks * g.waves;
}
template <int NP>
int64_t quad_slots(bool r64, const StageArgs &a) {
  return r64 ? quad_slots_epi<NP, false, 4>(a) : quad_slots_epi<NP, true, 3>(a);
}
template <bool CIN, int EPI>
void quad_orders(int np, const StageArgs &a, hipStream_t s) {
  switch (np) {
    case 4: quad_launch<4, CIN, EPI>(a, s); break;
    case 10: quad_launch<10, CIN, EPI>(a, s); break;
    case 20: quad_launch<20, CIN, EPI>(a, s); break;
    case 35: quad_launch<35, CIN, EPI>(a, s); break;
    default: throw Error{RFHIP_EUNSUPPORTED, "order not compiled (Np must be 4, 10, 20 or 35)"};
  }
  RF_HIP(hipGetLastError());
}

template <int NP, bool SEQ>
void quad_pack_np(const double *const D[3], const double *lift, std::vector<double> &out) {
  using Z = QuadSize<NP, SEQ>;
  constexpr int NG = QuadTab<NP>::NG, NFP = ElemTab<NP>::NFP, NFR = (Z::NF + 1) / 2;
  out.assign((size_t)NFR * 32, 0.0);
  // fragment t, row (contraction) kk, output i: pairs of fragments interleaved
  auto put = [&](int t, int kk, int i, double v) { out[(size_t)(t / 2) * 32 + (size_t)(4 * kk + i) * 2 + t % 2] = v; };
  int t = 0;
  for (int a = 0; a < NG; ++a)
    for (int b = 0; b < NG; ++b)
      for (int k = 0; k < 3; ++k) {
        if (!quad_nz<NP, SEQ>(k, a, b)) continue;
        for (int kk = 0; kk < 4; ++kk)
          for (int i = 0; i < 4; ++i) {
            const int r = quad_row<NP, SEQ>(a, i), c = quad_col<NP, SEQ>(b, kk);
            if (r < NP && c < NP) put(t, kk, i, D[k][r * NP + c]);
          }
        ++t;
      }
  // LIFT: the columns of step s are node s of every face, or (SEQ) four nodes
  // of one face in turn, the last step of a face filled up with zeros
  for (int s = 0; s < (SEQ ? 4 * Z::NU : NFP); ++s)
    for (int a = 0; a < NG; ++a, ++t)
      for (int kk = 0; kk < 4; ++kk) {
        const int f = SEQ ? s / Z::NU : kk, m = SEQ ? 4 * (s % Z::NU) + kk : s;
        for (int i = 0; i < 4; ++i) {
          const int r = quad_row<NP, SEQ>(a, i);
          if (r < NP && m < NFP) put(t, kk, i, lift[(size_t)r * 4 * NFP + f * NFP + m]);
        }
      }
}
// Whether every entry of D_k that is not 0.0 is one the SEQ kernels keep.
template <int NP>
bool quad_exact_np(const double *const D[3]) {
  for (int k = 0; k < 3; ++k)
    for (int i = 0; i < NP; ++i)
      for (int j = 0; j < NP; ++j)
        if (D[k][i * NP + j] != 0.0 && !((ElemTab<NP>::XM[k][i] >> j) & 1ull)) return false;
  return true;
}
template <int NP>
bool quad_pack_both(const double *const D[3], const double *lift, bool seq, std::vector<double> &out) {
  if (seq && !quad_exact_np<NP>(D)) return false;
  if (seq)
    quad_pack_np<NP, true>(D, lift, out);
  else
    quad_pack_np<NP, false>(D, lift, out);
  return true;
}
}  // namespace

bool quad_pack(int np, const double *const D[3], const double *lift, bool seq, std::vector<double> &out) {
  switch (np) {
    case 4: return quad_pack_both<4>(D, lift, seq, out);
    case 10: return quad_pack_both<10>(D, lift, seq, out);
    case 20: return quad_pack_both<20>(D, lift, seq, out);
    case 35: return quad_pack_both<35>(D, lift, seq, out);
    default: return false;
  }
}

void launch_quad(int np, int epi, const StageArgs &a, hipStream_t s) {
  switch (epi) {
    case 0: quad_orders<false, 0>(np, a, s); break;
    case 1: quad_orders<false, 1>(np, a, s); break;
    case 2: quad_orders<true, 2>(np, a, s); break;
    case 3: quad_orders<true, 3>(np, a, s); break;
    default: quad_orders<false, 4>(np, a, s); break;
  }
}

int64_t quad_kcl_slots(int np, bool r64, const StageArgs &a) {
  switch (np) {
    case 4: return quad_slots<4>(r64, a);
    case 10: return quad_slots<10>(r64, a);
    case 20: return quad_slots<20>(r64, a);
    case 35: return quad_slots<35>(r64, a);
    default: throw Error{RFHIP_EUNSUPPORTED, "the fused stage kernels run orders 1 to 4"};
  }
}

}  // namespace rfhip
