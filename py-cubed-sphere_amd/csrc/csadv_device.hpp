// Device-side helpers shared by the csadv kernels: descriptor layout, PPM edge
// reconstructions and the upwind flux.  gfx950 (CDNA4) only; 64-wide wavefronts.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "csadv.h"
#include "csadv_plan.hpp"

namespace csadv {

// A set of FP64 or dtype fields that receive a duo-grid ghost fill.
struct FieldSet {
  void *base[2];
  const int32_t *cur;        // device current-buffer index, or null (base[0])
  int32_t nfield, N, M, ld;
  int64_t fstride, pstride;
  const double *corr;        // per-field pending correction (null = none)
  const double *gc64;        // [M][ld] metric, used with corr
  const double *lagw;
  const int32_t *lagk;
  const int32_t *orient;
};

// Neighbour cell of the halo strip (panel p, side s) at depth d and along-edge index r.
// orient row = {q, ib, id, ir, jb, jd, jr}: i = ib + id*d + ir*r, j = jb + jd*d + jr*r.
__device__ __forceinline__ void halo_src(const int32_t *o, int d, int r, int &q, int &i, int &j) {
  q = o[0];
  i = o[1] + o[2] * d + o[3] * r;
  j = o[4] + o[5] * d + o[6] * r;
}

// Side of the neighbour across (p, side) and the sign relating the two axes across the edge.
// o = orient row {q, ib, id, ir, jb, jd, jr}; sides 0 E, 1 W, 2 N, 3 S.
__host__ __device__ inline void across(const int32_t *o, int side, int &sq, int &sign) {
  const int id = o[2], jd = o[5];
  sq = (id > 0) + (id == 0) * (2 + (jd > 0));       // id > 0: W; id < 0: E; id == 0: jd > 0 S, else N
  const int out = (side == 0 || side == 2) ? 1 : -1;
  const int in = (sq == 1 || sq == 3) ? 1 : -1;
  sign = out * in;
}

// Ghost target of (side, depth d, along-edge k); sides 0 E, 1 W, 2 N, 3 S.
// Written with selects, not a switch: where the side differs across a wavefront, hipcc
// (ROCm 7.2, gfx950) lowered the four-way switch so that the default arm's lanes kept a
// stale register for one of the two results.
__device__ __forceinline__ void ghost_target(int side, int d, int k, int N, int &i, int &j) {
  const int g = (side == 0 || side == 2) ? N + NG + d : NG - 1 - d;   // index across the side
  const bool xside = side < 2;
  i = xside ? g : k;
  j = xside ? k : g;
}

template <typename T> __device__ __forceinline__ T sgn(T x) { return (x > T(0)) ? T(1) : ((x < T(0)) ? T(-1) : T(0)); }

// x / B for a small constant B, with the division's own rounding in three operations (a division
// takes about ten): q is x times the rounded reciprocal, and one fma with the exact remainder
// x - B q corrects it (Markstein's theorem; checked against the division for every FP32 mantissa
// and 2e8 FP64 ones for B = 3, 6, 12).
template <int B, typename T>
__device__ __forceinline__ T div_const(T x) {
  const T y = T(1.0 / B), q = x * y;
  return __builtin_elementwise_fma(__builtin_elementwise_fma(T(-B), q, x), y, q);
}

// 1 / x, x near 1 (FP64): the hardware's estimate (24 bits) and two Newton steps, within an ulp.
__device__ __forceinline__ double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

// PPM edge values (q_L, q_R) of one cell from its 5-cell window; src/reconstruction_1d.py:26-193.
//   RECON 1 PPM-0 (CW84 eq. 1.9), 2 PPM-CW84 (monotone), 3 PPM-PL07 (eqs. 41-42), 4 PPM-L04 (B1-B4)
// The limited schemes (2: limited slopes at c-1, c, c+1, CW84 eqs. 1.7-1.8, a local extremum
// flattened, eq. 1.10, and overshoots cut; 4: monotone slopes, L04 eq. B1, edges by B3 and B4) as
// one text for two functions: limited_edges, whose multiply-adds the compiler fuses where it
// likes, and limited_edges_on, which fuses them within one source expression only, so that its bits do
// not depend on the kernel around it.
#define CSADV_LIMITED_EDGES(NAME, CONTRACT) \
template <typename T, int RECON> \
__device__ __forceinline__ void NAME(T m2, T m1, T c0, T p1, T p2, T &qL, T &qR) { \
  CONTRACT \
  if constexpr (RECON == 2) { \
 \
    auto slope = [](T a, T b, T c) { \
      T d0 = T(0.5) * (c - a), d1 = T(2.0) * (c - b), d2 = T(2.0) * (b - a); \
      T d = fmin(fabs(d0), fabs(d1)); \
      d = fmin(d, fabs(d2)) * sgn(d0); \
      return ((c - b) * (b - a) > T(0)) ? d : T(0); \
    }; \
    T sm = slope(m2, m1, c0), s0 = slope(m1, c0, p1), sp = slope(c0, p1, p2); \
    T R = T(0.5) * (p1 + c0) - div_const<6>(sp - s0); \
    T L = T(0.5) * (c0 + m1) - div_const<6>(s0 - sm); \
    T dq = R - L, q6 = T(6) * c0 - T(3) * (R + L); \
    if ((R - c0) * (c0 - L) <= T(0)) { R = c0; L = c0; } \
    bool over = fabs(dq) < fabs(q6); \
    T dd = R - L, mm = c0 - T(0.5) * (R + L); \
    const T d6 = div_const<6>(dd * dd); \
    bool left = dd * mm > d6; \
    bool right = -d6 > dd * mm; \
    if (over && left) L = T(3.0) * c0 - T(2.0) * R; \
    if (over && right) R = T(3.0) * c0 - T(2.0) * L; \
    qL = L; qR = R; \
  } else { \
 \
    auto mono = [](T a, T b, T c) { \
      T d = T(0.25) * (c - a); \
      T mx = fmax(fmax(a, b), c), mn = fmin(fmin(a, b), c); \
      return fmin(fmin(fabs(d), mx - b), b - mn) * sgn(d); \
    }; \
    T dm = mono(m2, m1, c0), d0 = mono(m1, c0, p1), dp = mono(c0, p1, p2); \
    T R = T(0.5) * (p1 + c0) - div_const<3>(dp - d0); \
    T L = T(0.5) * (c0 + m1) - div_const<3>(d0 - dm); \
    T s = sgn(T(2.0) * d0); \
    qL = c0 - fmin(T(2.0) * fabs(d0), fabs(L - c0)) * s; \
    qR = c0 + fmin(T(2.0) * fabs(d0), fabs(R - c0)) * s; \
  } \
}
CSADV_LIMITED_EDGES(limited_edges, )
CSADV_LIMITED_EDGES(limited_edges_on, _Pragma("clang fp contract(on)"))
#undef CSADV_LIMITED_EDGES

template <typename T, int RECON>
__device__ __forceinline__ void recon_edges(T m2, T m1, T c0, T p1, T p2, T &qL, T &qR) {
  if constexpr (RECON == 3) {
    const T a1 = T(2.0 / 60.0), a2 = T(-13.0 / 60.0), a3 = T(47.0 / 60.0), a4 = T(27.0 / 60.0), a5 = T(-3.0 / 60.0);
    qR = a1 * m2 + a2 * m1 + a3 * c0 + a4 * p1 + a5 * p2;
    qL = a5 * m2 + a4 * m1 + a3 * c0 + a2 * p1 + a1 * p2;
  } else if constexpr (RECON == 1) {
    const T s7 = T(7.0 / 12.0);
    qR = s7 * (p1 + c0) - div_const<12>(p2 + m1);
    qL = s7 * (c0 + m1) - div_const<12>(p1 + m2);
  } else {
    limited_edges<T, RECON>(m2, m1, c0, p1, p2, qL, qR);
  }
}

// The parabola of one cell as the upwind flux uses it (src/flux.py:28-44): edge values
// from the 5-cell window, with the MT-0 metric applied (gl / gr at the cell's left and right
// edges, gcell at its centre).  With dq = q_R - q_L and q6 = 6q - 3(q_R + q_L), it is kept in
// the scaled form the flux below evaluates fastest: with a = 3q - (q_R + q_L),
//   rB = a - q_R = (q6 - dq) / 2,   lB = a - q_L = (q6 + dq) / 2,   q6' = a - q = q6 / 3.
// An edge takes it from the cell on its left when the wind there is non-negative
// (A = q_R, B = rB) and from the cell on its right otherwise (A = q_L, B = -lB).  Each cell's
// parabola is formed once and an edge only selects three values from one side.
template <typename T>
struct Parab {
  T rA, rB, lA, lB, q6;
};

// The parabola from a cell's edge values (q_L, q_R) and mean c0.
template <typename T>
__device__ __forceinline__ Parab<T> parab_of(T qL, T qR, T c0, T gl, T gr, T gcell, bool mt0) {
  T q = c0;
  if (mt0) { qL = qL * gl; qR = qR * gr; q = q * gcell; }
  const T a = T(3) * q - (qR + qL);
  return {qR, a - qR, qL, a - qL, a - q};
}

template <typename T, int RECON>
__device__ __forceinline__ Parab<T> parabola(T m2, T m1, T c0, T p1, T p2, T gl, T gr, T gcell, bool mt0) {
  T qL, qR;
  recon_edges<T, RECON>(m2, m1, c0, p1, p2, qL, qR);
  return parab_of<T>(qL, qR, c0, gl, gr, gcell, mt0);
}

// Upwind PPM flux through one edge (src/flux.py:48-70) from the parabolas of the cells on its
// left (L) and right (R): f = q_R + (c/2)(q6 - dq) - q6 c^2/3 from the left cell when up,
// f = q_L - (c/2)(q6 + dq) - q6 c^2/3 from the right cell otherwise; F = f u_avg, and
// MT-PL07 multiplies by the edge metric ge.  Returned already times dt/dx, as F dt/dx =
// f c (c = u_avg dt/dx, the Courant number), so the flux difference of a cell is the
// difference of two returned values.  In the scaled form of the parabola,
// f = A + c (B - q6' c): three operations with the final product by c.
template <typename T>
__device__ __forceinline__ T upwind(bool up, T LrA, T LrB, T Lq6, const Parab<T> &R, T cc, T ge, bool mt0) {
  const T A = up ? LrA : R.lA, B = up ? LrB : -R.lB, q6 = up ? Lq6 : R.q6;
  T f = (A + cc * (B - q6 * cc)) * cc;
  if (!mt0) f = f * ge;
  return f;
}

// Upwind flux in weighted form.  With c the Courant number of an edge, s = c when the wind there
// is non-negative and -c otherwise, A the upwind cell's edge value at this edge, D its other edge
// value and q its mean (A, D, q with the MT-0 metric on them), CW84's flux (src/flux.py:28-70) is
//   F dt/dx = c (al A + be D + ga q),  al = (1 - s)^2,  be = -s (1 - s),  ga = s (3 - 2 s),
// so every edge is three products with weights that depend on the wind and the metric only: they
// are formed once per edge and serve both passes of the split and every tracer.
// PPM-0 and PPM-PL07 are linear in the window, so their edge values split into a part symmetric
// and a part antisymmetric about the cell, A, D = e +- o, with
//   e = k3 q + k1 (S1 + r S2),  o = h1 (D1 + t D2),  S, D the sums and differences of the
// neighbours at distance 1 and 2: a cell is then six operations (where its two edge values and
// their parabola took eighteen) and k1, k3, h1 go into the weights.
template <int RECON> struct Lin {
  static constexpr bool on = RECON == 1 || RECON == 3;
  static constexpr double k3 = RECON == 1 ? 7.0 / 12.0 : 47.0 / 60.0, k1 = RECON == 1 ? 0.25 : 14.0 / 120.0;
  static constexpr double r = RECON == 1 ? -1.0 / 6.0 : -1.0 / 14.0, h1 = 1.0 / 3.0, t = -1.0 / 8.0;
};

// What an edge takes from a cell: linear schemes a = S1 + r S2, b = D1 + t D2, the others the edge
// values a = q_L, b = q_R; q the mean.
template <typename T>
struct Cell {
  T a, b, q;
};

template <typename T, int RECON>
__device__ __forceinline__ Cell<T> cell_of(T m2, T m1, T c0, T p1, T p2) {
  using L = Lin<RECON>;
  Cell<T> c;
  c.q = c0;
  if constexpr (L::on) {
    c.a = __builtin_elementwise_fma(T(L::r), p2 + m2, p1 + m1);
    c.b = __builtin_elementwise_fma(T(L::t), p2 - m2, p1 - m1);
  } else {
    limited_edges_on<T, RECON>(m2, m1, c0, p1, p2, c.a, c.b);
  }
  return c;
}

// An edge's weights: of the upwind cell's mean (w0) and, linear schemes, its a and b (w1, w2), the
// others its A and D; up: the upwind cell is the left one.
template <typename T>
struct EdgeW {
  T w0, w1, w2;
  bool up;
};

// An edge's entry in a flux table: w0, w1, w2 and, with four words, its metric-weighted Courant
// number h (the splittings' dc = c1 - c2).  The side of the upwind cell is the lowest bit of w2:
// that moves w2, the weight of the window's antisymmetric part (or of the far edge value), by
// less than an ulp, where its sign or a separate wind would cost another load and compare.
template <typename T>
struct FluxEntry {
  T w0, w1, w2, h;
};
__device__ __forceinline__ double tag_low(double v, bool b) {
  return __longlong_as_double((__double_as_longlong(v) & ~1ll) | (b ? 1ll : 0ll));
}
__device__ __forceinline__ bool low_tag(double v) { return (unsigned)__double_as_longlong(v) & 1u; }

// The weights of an edge with Courant number c (s as above), gA / gD the edge metrics at the edge
// and at the upwind cell's other edge, gq its centre metric (MT-0); MT-PL07 (mt0 false) takes the
// edge's metric gA on the whole flux.  Multiply-adds are written as fma where they fuse and the
// compiler fuses no others (here and in the march), so that the bits do not depend on the
// surrounding code: a solve alone and in a batch, and its weights formed in the step or read from
// a table, agree.
template <typename T, int RECON>
__device__ __forceinline__ EdgeW<T> edge_weights(bool up, T c, T s, T gA, T gD, T gq, bool mt0) {
#pragma clang fp contract(off)
  using L = Lin<RECON>;
  const T om = T(1) - s, ga = s * __builtin_elementwise_fma(T(-2), s, T(3));
  EdgeW<T> w;
  w.up = up;
  if (mt0) {
    const T ag = (om * om) * gA, t = s * om;
    if constexpr (L::on) {
      const T P = __builtin_elementwise_fma(-t, gD, ag), M = __builtin_elementwise_fma(t, gD, ag);
      w.w0 = c * __builtin_elementwise_fma(T(L::k3), P, ga * gq);
      w.w1 = (c * T(L::k1)) * P;
      w.w2 = (s * T(L::h1)) * M;
    } else {
      w.w0 = c * (ga * gq);
      w.w1 = c * ag;
      w.w2 = -c * (t * gD);
    }
  } else {
    const T cg = c * gA;
    if constexpr (L::on) {
      const T P = om * (om - s);
      w.w0 = cg * __builtin_elementwise_fma(T(L::k3), P, ga);
      w.w1 = (cg * T(L::k1)) * P;
      w.w2 = ((s * gA) * T(L::h1)) * om;
    } else {
      w.w0 = cg * ga;
      w.w1 = cg * (om * om);
      w.w2 = -cg * (s * om);
    }
  }
  w.w2 = tag_low(w.w2, up);   // (as a table holds it)
  return w;
}

// Flux (times dt/dx) of an edge from the cells on its left and right.
template <typename T, int RECON>
__device__ __forceinline__ T edge_flux(const EdgeW<T> &w, T la, T lb, T lq, const Cell<T> &R) {
  constexpr bool lin = Lin<RECON>::on;
  const T q = w.up ? lq : R.q, x = w.up ? (lin ? la : lb) : R.a, y = w.up ? (lin ? lb : la) : R.b;
  return __builtin_elementwise_fma(w.w2, y, __builtin_elementwise_fma(w.w1, x, w.w0 * q));
}

// Whole-wavefront DPP lane shifts (one v_mov_b32_dpp per dword, no LDS round trip):
// from_left(v) is v of lane-1, from_right(v) is v of lane+1; the end lane without a source
// (lane 0, resp. lane 63) reads zero.  The step kernel only ever stores results of lanes
// whose stencils stay at least two lanes away from either end, so the end values never
// reach a stored cell.
constexpr int kDppWaveShl1 = 0x130;   // lane i <- lane i+1
constexpr int kDppWaveShr1 = 0x138;   // lane i <- lane i-1
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
template <typename T> __device__ __forceinline__ T from_left(T v) { return dpp_move<kDppWaveShr1>(v); }
template <typename T> __device__ __forceinline__ T from_right(T v) { return dpp_move<kDppWaveShl1>(v); }

// Lane pull through the LDS crossbar (ds_bpermute_b32: no LDS memory, no VALU slot): each lane
// reads v of the lane whose byte address (4 * lane) it passes; the address wraps modulo 64 lanes.
__device__ __forceinline__ float lane_pull(float v, int addr) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(v)));
}
__device__ __forceinline__ double lane_pull(double v, int addr) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_ds_bpermute(addr, (int)b);
  const int hi = __builtin_amdgcn_ds_bpermute(addr, (int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// The 5-cell window of every lane's cell along the wavefront (x): neighbours at -2, -1, +1, +2.
// PULL: through the crossbar (am2 / am1 / ap1 / ap2: byte addresses of the lanes two and one to
// the left and right, mod 64), which frees four VALU slots per window and adds the crossbar's
// latency; else by DPP shifts.  End lanes read zeros (DPP) or wrapped lanes (crossbar); no
// stored cell's stencil reaches them.
template <typename T, bool PULL>
__device__ __forceinline__ void xwindow(T v, int am2, int am1, int ap1, int ap2, T &m2, T &m1, T &p1, T &p2) {
  if constexpr (PULL) {
    m2 = lane_pull(v, am2); m1 = lane_pull(v, am1);
    p1 = lane_pull(v, ap1); p2 = lane_pull(v, ap2);
  } else {
    m1 = from_left(v); p1 = from_right(v);
    m2 = from_left(m1); p2 = from_right(p1);
  }
}

// Flux through the left edge of each lane's cell along the wavefront (x), lane = cell: every
// lane forms the flux its cell sends through its right edge when it is the upwind cell there
// (c_r = c of the right neighbour) and through its left edge when it is the upwind cell there;
// the left edge then takes the left neighbour's right-edge value when the wind there is
// non-negative and the lane's own value otherwise.  One shift of the result replaces shifting
// the left cell's three parabola values (the same arithmetic as upwind(), so the same bits).
// gl, gr: edge metrics at the left and right edges (MT-PL07 only).
template <typename T>
__device__ __forceinline__ T upwind_x(bool up, const Parab<T> &c, T cc, T gl, T gr, bool mt0) {
  const T ccr = from_right(cc);
  T fr = (c.rA + ccr * (c.rB - c.q6 * ccr)) * ccr;
  T fl = (c.lA + cc * (-c.lB - c.q6 * cc)) * cc;
  if (!mt0) { fr = fr * gr; fl = fl * gl; }
  const T from_l = from_left(fr);
  return up ? from_l : fl;
}

// Flux through the left edge of each lane's cell along the wavefront (x): the left cell's a and b
// by lane shifts, its mean from the window (m1).
template <typename T, int RECON>
__device__ __forceinline__ T edge_flux_x(const EdgeW<T> &w, const Cell<T> &c, T m1) {
  return edge_flux<T, RECON>(w, from_left(c.a), from_left(c.b), m1, c);
}

// Element idx of an array whose base is wave-uniform: the byte offset stays 32-bit so that
// the load takes the scalar-base + vector-offset form (callers keep idx * sizeof(T) < 4 GiB).
// Every array handed to the library is device global memory, so the access is made in the
// global address space (a generic pointer would compile to a flat access).
#define CSADV_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ T ld_at(const T *base, uint32_t idx) {
  const char CSADV_GLOBAL *b = (const char CSADV_GLOBAL *)(base);
  return *(const T CSADV_GLOBAL *)(b + idx * (uint32_t)sizeof(T));
}
template <typename T>
__device__ __forceinline__ void st_at(T *base, uint32_t idx, T v) {
  char CSADV_GLOBAL *b = (char CSADV_GLOBAL *)(base);
  *(T CSADV_GLOBAL *)(b + idx * (uint32_t)sizeof(T)) = v;
}

// Stores that every lane issues, with no branch around them: a lane with nothing to store passes
// an offset past the buffer's end, and the buffer's range check drops its write.  Used where a
// branch would make the count of outstanding memory operations uncertain: loads and stores share
// one counter, and a wait for a load past an optional store has to assume the store was not
// issued, waiting for that much more than it needs.  The buffer covers `bytes` bytes from `base`
// (< 2^31); kNoStore is past the end of any such buffer.
constexpr uint32_t kNoStore = 0x80000000u;
constexpr int kBufferDword3 = 0x00020000;   // raw (untyped) 32-bit elements, no swizzle
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(base, (short)0, (int)bytes, kBufferDword3);
}
typedef unsigned int csadv_u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void st_buf(__amdgpu_buffer_rsrc_t r, uint32_t byte_off, double v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(csadv_u32x2, v), r, byte_off, 0, 0);
}
__device__ __forceinline__ void st_buf(__amdgpu_buffer_rsrc_t r, uint32_t byte_off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned int, v), r, byte_off, 0, 0);
}

// Entry at byte offset off of a flux table (buffer loads: three words at once need no alignment
// padding; the buffer covers one panel's table, under 2^32 bytes).
template <int NW>
__device__ __forceinline__ FluxEntry<double> ld_flux(__amdgpu_buffer_rsrc_t r, uint32_t off, double) {
  typedef double f64x2 __attribute__((ext_vector_type(2)));
  const f64x2 a = __builtin_bit_cast(f64x2, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  if constexpr (NW == 3) {
    return {a.x, a.y, __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 16, 0)), 0.0};
  } else {
    const f64x2 b = __builtin_bit_cast(f64x2, __builtin_amdgcn_raw_buffer_load_b128(r, off, 16, 0));
    return {a.x, a.y, b.x, b.y};
  }
}

// The wind of one edge from a one-field basis W and its coefficient s at the step's time
// (src/averaged_velocity.py:14-62 with RK1: the wind at t_n), in FP64, in one expression shared by
// the wind kernel and the step kernel so that both give the same bits (s = 1 gives w, with a
// zero of either sign as +0).
__device__ __forceinline__ double wind_of_basis(double s, double w) { return fma(s, w, 0.0); }

// Split update of one cell after the first directional pass (src/discrete_operators.py:49-73).
//   split 1 AVLT: (gQ + dF/2)/g ; 2 L04: (gQ + dF/2 + (c1-c2) Q/2)/g ; 3 PL07: (Q + (Q+dF)/(1-(c1-c2)))/2
template <typename T>
__device__ __forceinline__ T split_update(int split, T Q, T dF, T g, T rg, T c1, T c2) {
  if (split == 1) return (Q * g + T(0.5) * dF) * rg;
  if (split == 2) return (Q * g + T(0.5) * dF + T(0.5) * (c1 - c2) * Q) * rg;
  if constexpr (!std::is_same<T, float>::value) return T(0.5) * (Q + (Q + dF) * recip(T(1.0) - (c1 - c2)));
  else return T(0.5) * (Q + (Q + dF) / (T(1.0) - (c1 - c2)));
}

// The split's half-step of one cell (src/discrete_operators.py:49-73) in two parts: a factor that
// depends on the winds and the metric only (shared by the tracers), and the update with it.
// dc = c1 - c2, the difference of the metric-weighted Courant numbers of the cell's edges.
//   AVLT: Q + dF / (2 g);  L04: Q + (dF + dc Q) / (2 g);  PL07: Q / 2 + (Q + dF) / (2 (1 - dc))
template <typename T, int SPLIT>
__device__ __forceinline__ T half_factor(T rg, T dc) {
#pragma clang fp contract(off)
  if constexpr (SPLIT == 3) return T(0.5) * recip(T(1) - dc);
  else return T(0.5) * rg;
}
template <typename T, int SPLIT>
__device__ __forceinline__ T half_step(T Q, T dF, T h, T dc) {
#pragma clang fp contract(off)
  if constexpr (SPLIT == 1) return __builtin_elementwise_fma(h, dF, Q);
  else if constexpr (SPLIT == 2) return __builtin_elementwise_fma(h, __builtin_elementwise_fma(dc, Q, dF), Q);
  else return __builtin_elementwise_fma(h, Q + dF, T(0.5) * Q);
}
__device__ __forceinline__ float fabs_t(float v) { return fabsf(v); }
__device__ __forceinline__ double fabs_t(double v) { return fabs(v); }

// MF-AF (src/edges_treatment.py:231-278) on boundary cells of a new state: F holds the second
// pass's fluxes through the 24 panel sides ([panel][E, W, N, S][N], scaled by dt/dx as the step
// forms them); each is replaced by the average of the two panels' fluxes through that cube edge,
// 0.5 f + 0.5 (sign f'), with the neighbour's side and sign from the halo orientation table, by
// adding the difference to the boundary cells: Q += (f - f_avg) / g at the east and north sides
// (their fluxes leave the cell there) and (f_avg - f) / g at the west and south sides.  Item idx
// is one boundary cell of a panel (4 (N - 1) of them per panel), so a corner cell takes both of
// its sides' differences in one fixed order; run is the step that produced the state.
// Where the flux across (panel, side) at position k lies: index a + k b of F, and the sign.
struct AfSide {
  int32_t a, b, sign;
};
__host__ __device__ inline AfSide af_side(const int32_t *o, int side, int N) {
  // o: the side's orientation row {q, ib, id, ir, jb, jd, jr}, here at depth 0 and row k + NG
  int sq, sign;
  across(o, side, sq, sign);
  const int along0 = sq < 2 ? o[4] + o[6] * NG : o[1] + o[3] * NG;
  return {(o[0] * 4 + sq) * N + along0 - NG, sq < 2 ? o[6] : o[3], sign};
}

struct AfSides {
  AfSide side[24];
};

// The grid's x covers the panels' rings, panel by panel (af_blocks blocks each), so that the panel is
// wave-uniform and its sides' places are scalar loads.  side_of(p, side): the AfSide of a panel side,
// from the orientation table or from kernel arguments (a chain of loads less).
inline int af_blocks(int N) { return (4 * (N - 1) + BLOCK - 1) / BLOCK; }
template <typename T, typename SideOf>
__device__ __forceinline__ void af_fix_cell(const Solve &S, int tr, int run, const T *F, SideOf side_of) {
  const csadv_solve_desc &D = S.d;
  const int N = D.N, ld = D.ld, i0 = NG, iend = N + NG;
  const int per = gridDim.x / 6, p = blockIdx.x / per, c = (blockIdx.x - p * per) * BLOCK + threadIdx.x;
  const AfSide sides[4] = {side_of(p, 0), side_of(p, 1), side_of(p, 2), side_of(p, 3)};
  if (c >= 4 * (N - 1)) return;
  int i, j;
  // ring order: south row, north row, west column, east column (corners in the rows)
  if (c < N) { i = i0 + c; j = i0; }
  else if (c < 2 * N) { i = i0 + c - N; j = iend - 1; }
  else if (c < 3 * N - 2) { i = i0; j = i0 + 1 + c - 2 * N; }
  else { i = iend - 1; j = i0 + 1 + c - (3 * N - 2); }
  const auto average = [&](int side, int k) {
    const AfSide f = sides[side];
    const T own = F[(p * 4 + side) * N + k], nb = F[f.a + f.b * k];
    return T(0.5) * own + T(0.5) * (f.sign > 0 ? nb : -nb);
  };
  T d = T(0);
  if (i == iend - 1) d += F[(p * 4 + 0) * N + j - NG] - average(0, j - NG);
  if (i == i0) d += average(1, j - NG) - F[(p * 4 + 1) * N + j - NG];
  if (j == iend - 1) d += F[(p * 4 + 2) * N + i - NG] - average(2, i - NG);
  if (j == i0) d += average(3, i - NG) - F[(p * 4 + 3) * N + i - NG];
  T *Q = reinterpret_cast<T *>(((run + 1) & 1) ? D.q1 : D.q0) + tr * S.tstride + p * S.pstride;
  const T rg = reinterpret_cast<const T *>(D.rgc)[(int64_t)j * ld + i];
  Q[(int64_t)j * ld + i] += d * rg;
}

// Bring every cache line of the kernel-argument descriptor into the scalar cache with loads
// issued together: an empty asm takes one word of each line and passes v through unchanged, so
// v exists only once all of them have arrived (one scalar round trip); the field loads at their
// first use then hit the cache instead of waiting for their lines one after another (the
// one-solve step kernel's start took four such dependent round trips).  The asm is neither
// volatile nor a memory clobber, so the loads after it may still be scalar loads.  (For a
// descriptor in global memory the compiler reads the words with vector loads, which warm no
// scalar cache: the multi-solve kernel does not use it.)
__device__ __forceinline__ int touch_solve(const Solve &S, int v) {
  static_assert(sizeof(Solve) == 448, "one word in each 64-byte line of the descriptor");
  const char *b = reinterpret_cast<const char *>(&S);
  int w[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) __builtin_memcpy(&w[k], b + (k < 7 ? 64 * k : 444), 4);
  asm("" : "=s"(v) : "0"(v), "s"(w[0]), "s"(w[1]), "s"(w[2]), "s"(w[3]), "s"(w[4]), "s"(w[5]), "s"(w[6]), "s"(w[7]));
  return v;
}

// Sum over a wavefront, complete in lane 0, in the order of shuffles down by 32, 16, 8, 4, 2, 1:
// the halves and the rows of 16 by gfx950's lane swaps, within a row by DPP shifts (a tenth of the
// latency of shuffles through the LDS crossbar, on the critical path at both ends of a march).
__device__ __forceinline__ double lane_up32(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
  const unsigned l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false)[1];
  const unsigned h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false)[1];
  return __longlong_as_double(((long long)h << 32) | l);
}
__device__ __forceinline__ double lane_up16(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
  const unsigned l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false)[1];
  const unsigned h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false)[1];
  return __longlong_as_double(((long long)h << 32) | l);
}
__device__ __forceinline__ double warp_sum(double v) {
  v += lane_up32(v);
  v += lane_up16(v);
  v += dpp_move<0x108>(v);   // row_shl:8 -- lane i takes lane i + 8 of its row
  v += dpp_move<0x104>(v);
  v += dpp_move<0x102>(v);
  v += dpp_move<0x101>(v);
  return v;
}
// The same, in every lane.
__device__ __forceinline__ double wave_total(double v) {
  const long long b = __double_as_longlong(warp_sum(v));
  const int lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Mass-fixer correction total C after `steps` steps, from the stored totals c0 / c1 (slots of
// even / odd steps) and the partials' sum: with the partials of the last step pending,
// C = C(steps - 1) + dt m0 / a2, m0 = sum of div g over the interior
// (src/discrete_operators.py:98-101); otherwise C is the stored total of this step.
__device__ __forceinline__ double corr_total(double dt, double a2, double c0, double c1, double sum, int pending,
                                             int steps) {
  const double held = (steps & 1) ? c1 : c0, prev = (steps & 1) ? c0 : c1;
  return pending ? prev + dt * sum / a2 : held;
}

// A strip ghost's value: its four sources in recipe order, every product fused.
__device__ __forceinline__ double strip_sum(double v0, double v1, double v2, double v3, double w0, double w1, double w2,
                                            double w3) {
  return fma(v3, w3, fma(v2, w2, fma(v1, w1, v0 * w0)));
}

// Row m (0 .. 5) of the corner ghosts outside a panel: the three below it, the three above.
__device__ __forceinline__ int corner_row(int m, int N) { return m < 3 ? NG - 3 + m : N + NG + m - 3; }

}  // namespace csadv
