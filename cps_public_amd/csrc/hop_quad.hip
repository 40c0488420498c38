// The half-precision hop with the SU(3) products on the matrix cores, for
// layouts that keep at least four spinors of one site side by side (the
// Ls/2 slots of a domain-wall field, the Ls slices of a Moebius field; nb a
// multiple of 4).
//
// v_mfma_f32_4x4x4_16b_f16 multiplies 16 independent 4x4 blocks, one per
// group of 4 lanes: lane 4b + i holds row i of A and column i of B, and gets
// column i of the product.  Here the four lanes of a group are four slots of
// one site, so A is the site's link (lane i loads row i, 12 bytes, instead
// of every lane loading all 36) and column i is the projected half spinor of
// lane i's own slot: operands and results never move between lanes.  A
// direction takes 8 instructions, (2 spins) x (real, imaginary part) x (two
// halves of the colour sum); the FP16 products and FP32 sums are those of
// v_dot2_f32_f16, which takes 36 per direction, and the matrix cores run
// beside the vector ALU.
//
// The links are stored once per output site and direction (pack_gauge_quad):
// the 8 links that the hop onto a site uses lie next to each other, the
// backward ones daggered, so every lane reads its rows at immediate
// offsets from one address.  BF16 links are kept as the FP16 numbers that
// the product uses.
//
// The element kernel issues ~900 vector instructions per wavefront here and
// keeps the vector ALUs 55-60% busy; this one issues ~570 and 64 matrix
// instructions, and is bound by the vector L1's data return and outstanding
// misses: with the field in HBM the return path is busy 97% of the launch and
// a CU has 59-82 lines in flight at 450-640 clocks, 10 TB/s from L2 over the
// chip (16^3x32, Moebius, Ls 16, 12 rhs); with one rhs of a domain-wall field
// 49-57 lines at 315-420 clocks while the CUs are busy 77-82% of a launch of
// 36-55 us (profiles/performance_cases_hop_counters.txt).  One hop of the
// 16^3x32 lattice takes 452 instead of 488 us (Moebius, Ls 16, 12 rhs) and,
// with the sites swept block by block (HOP_SPATIAL), 38 instead of 46 us
// (domain wall, Ls 16, 1 rhs).
//
// Neighbour loads run CPSHIP_QUAD_AHEAD directions ahead of the arithmetic:
// 5 directions at 3 waves per SIMD measured best (3 at 4 waves 466 us, 6 at
// 3 451, 8 at 2 455; 2 at 5 waves spills, 742).
#include "hop_kernel.h"

namespace cpship {

typedef _Float16 hv4 __attribute__((ext_vector_type(4)));
typedef float fv4 __attribute__((ext_vector_type(4)));

#ifndef CPSHIP_QUAD_AHEAD
#define CPSHIP_QUAD_AHEAD 5
#endif
#ifndef CPSHIP_QUAD_WAVES
#define CPSHIP_QUAD_WAVES 3
#endif

// epilogues: out = scale hop, out = xcoef X + scale hop, the fused Moebius
// stages (see hop_kernel.h), and the residual updates
enum { QE_PLAIN = 0, QE_M5 = 1, QE_S5X = 2, QE_S5XR = 3, QE_S5XRR = 4, QE_NRR = 5, QE_X = 6 };

struct QuadDir {
  uint4 q[3];
  float n;
  uint32_t w[3];
};

struct QuadSite {
  uint32_t idx[8];      // neighbour sites
  uint32_t e0;          // 16 * (element of slot j at neighbour site 0)
  uint32_t stride;      // 16 * nb
  const char* links;    // row min(lane & 3, 2) of the site's first link
};

template <int D>
__device__ __forceinline__ void quad_load(const HopParams& P, const QuadSite& Q, QuadDir& r) {
  const uint32_t off = Q.e0 + __umul24(Q.idx[D], Q.stride);
  const int64_t pb = P.in.plane * 16;
#pragma unroll
  for (int k = 0; k < 3; k++) r.q[k] = ld_off<uint4>(P.in.data, k * pb, off);
  r.n = ld_off<float>(P.in.norm, 0, off >> 2);
  const uint32_t* l = reinterpret_cast<const uint32_t*>(Q.links + 36 * D);
#pragma unroll
  for (int k = 0; k < 3; k++) r.w[k] = l[k];
}

// h = p + alpha q (alpha = +1, -1, +i, -i for ALPHA = 0..3, see ProjAlpha):
// one v_pk_add_f16, the half selection and the signs are its modifiers
template <int ALPHA>
__device__ __forceinline__ hv2 proj_pair(hv2 p, hv2 q) {
  if constexpr (ALPHA == 0) return p + q;
  else if constexpr (ALPHA == 1) return p - q;
  else if constexpr (ALPHA == 2) return p + hv2{-q.y, q.x};
  else return p + hv2{q.y, -q.x};
}

// (im, re) of a link word (re, -im)
__device__ __forceinline__ hv2 link_im(hv2 w) { return hv2{-w.y, w.x} + hv2{(_Float16)0, (_Float16)0}; }

__device__ __forceinline__ hv4 pair4(hv2 a, hv2 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3); }

template <int D, int DAG>
__device__ __forceinline__ void quad_compute(const QuadDir& r, cplx<float> acc[12]) {
  constexpr int MU = D & 3;
  constexpr int S = (DAG == 0) ? 1 : -1;
  constexpr int A = (D < 4) ? -S : S;
  using PA = ProjAlpha<MU, A>;
  const hv2 p[12] = {as_hv2(r.q[0].x), as_hv2(r.q[0].y), as_hv2(r.q[0].z), as_hv2(r.q[0].w),
                     as_hv2(r.q[1].x), as_hv2(r.q[1].y), as_hv2(r.q[1].z), as_hv2(r.q[1].w),
                     as_hv2(r.q[2].x), as_hv2(r.q[2].y), as_hv2(r.q[2].z), as_hv2(r.q[2].w)};
  hv2 h0[3], h1[3];   // projected spins 0, 1
#pragma unroll
  for (int c = 0; c < 3; c++) {
    h0[c] = proj_pair<PA::a0>(p[c], p[3 * PA::q0 + c]);
    h1[c] = proj_pair<PA::a1>(p[3 + c], p[3 * PA::q1 + c]);
  }
  // (re, -im) . (h.re, h.im) is the real part of a product, (im, re) . h the
  // imaginary one; colours 0, 1 fill one K = 4 operand, colour 2 half of
  // another (its other half is zero in the spinor operand)
  const hv2 u[3] = {as_hv2(r.w[0]), as_hv2(r.w[1]), as_hv2(r.w[2])};
  const hv2 v[3] = {link_im(u[0]), link_im(u[1]), link_im(u[2])};
  const hv2 z2 = {(_Float16)0, (_Float16)0};
  const hv4 u01 = pair4(u[0], u[1]), v01 = pair4(v[0], v[1]), u2 = pair4(u[2], v[2]), v2 = pair4(v[2], u[2]);
  const hv4 a01 = pair4(h0[0], h0[1]), b01 = pair4(h1[0], h1[1]), a2 = pair4(h0[2], z2), b2 = pair4(h1[2], z2);
  const fv4 z = {0.f, 0.f, 0.f, 0.f};
  fv4 w0[2], w1[2];
  w0[0] = __builtin_amdgcn_mfma_f32_4x4x4f16(u01, a01, z, 0, 0, 0);
  w0[1] = __builtin_amdgcn_mfma_f32_4x4x4f16(v01, a01, z, 0, 0, 0);
  w1[0] = __builtin_amdgcn_mfma_f32_4x4x4f16(u01, b01, z, 0, 0, 0);
  w1[1] = __builtin_amdgcn_mfma_f32_4x4x4f16(v01, b01, z, 0, 0, 0);
  w0[0] = __builtin_amdgcn_mfma_f32_4x4x4f16(u2, a2, w0[0], 0, 0, 0);
  w0[1] = __builtin_amdgcn_mfma_f32_4x4x4f16(v2, a2, w0[1], 0, 0, 0);
  w1[0] = __builtin_amdgcn_mfma_f32_4x4x4f16(u2, b2, w1[0], 0, 0, 0);
  w1[1] = __builtin_amdgcn_mfma_f32_4x4x4f16(v2, b2, w1[1], 0, 0, 0);
  // acc += n (full spinor rebuilt from w), each sum one fused multiply-add
  const float n = r.n, an = A * r.n;
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const float ar = w0[0][c], ai = w0[1][c], br = w1[0][c], bi = w1[1][c];
    acc[c].re = fmaf(n, ar, acc[c].re);
    acc[c].im = fmaf(n, ai, acc[c].im);
    acc[3 + c].re = fmaf(n, br, acc[3 + c].re);
    acc[3 + c].im = fmaf(n, bi, acc[3 + c].im);
    if constexpr (MU == 0) {          // r2 = -A i w1, r3 = -A i w0
      acc[6 + c].re = fmaf(an, bi, acc[6 + c].re);
      acc[6 + c].im = fmaf(-an, br, acc[6 + c].im);
      acc[9 + c].re = fmaf(an, ai, acc[9 + c].re);
      acc[9 + c].im = fmaf(-an, ar, acc[9 + c].im);
    } else if constexpr (MU == 1) {   // r2 = A w1, r3 = -A w0
      acc[6 + c].re = fmaf(an, br, acc[6 + c].re);
      acc[6 + c].im = fmaf(an, bi, acc[6 + c].im);
      acc[9 + c].re = fmaf(-an, ar, acc[9 + c].re);
      acc[9 + c].im = fmaf(-an, ai, acc[9 + c].im);
    } else if constexpr (MU == 2) {   // r2 = -A i w0, r3 = A i w1
      acc[6 + c].re = fmaf(an, ai, acc[6 + c].re);
      acc[6 + c].im = fmaf(-an, ar, acc[6 + c].im);
      acc[9 + c].re = fmaf(-an, bi, acc[9 + c].re);
      acc[9 + c].im = fmaf(an, br, acc[9 + c].im);
    } else {                          // r2 = A w0, r3 = A w1
      acc[6 + c].re = fmaf(an, ar, acc[6 + c].re);
      acc[6 + c].im = fmaf(an, ai, acc[6 + c].im);
      acc[9 + c].re = fmaf(an, br, acc[9 + c].re);
      acc[9 + c].im = fmaf(an, bi, acc[9 + c].im);
    }
  }
}

// v += c * (n h) for the two halves of word w (n h is exact in the fused
// multiply-add up to the one rounding of c n)
__device__ __forceinline__ void fma_word(uint32_t w, float cn, cplx<float>& v) {
  const hv2 h = as_hv2(w);
  v.re = fmaf(float(h.x), cn, v.re);
  v.im = fmaf(float(h.y), cn, v.im);
}

// a half spinor (components c0 .. c0+5) as words, and its norm
__device__ __forceinline__ void load_half_words(const FieldRef& f, uint32_t e, int c0, uint32_t w[6], float& n) {
  const int64_t pb = f.plane * 16;
  if (c0 == 0) {
    const uint4 q = ld_off<uint4>(f.data, 0, e << 4);
    const uint2 r = ld_off<uint2>(f.data, pb, e << 4);
    w[0] = q.x; w[1] = q.y; w[2] = q.z; w[3] = q.w; w[4] = r.x; w[5] = r.y;
  } else {
    const uint2 r = ld_off<uint2>(f.data, pb + 8, e << 4);
    const uint4 q = ld_off<uint4>(f.data, 2 * pb, e << 4);
    w[0] = r.x; w[1] = r.y; w[2] = q.x; w[3] = q.y; w[4] = q.z; w[5] = q.w;
  }
  n = ld_off<float>(f.norm, 0, e << 2);
}

__device__ __forceinline__ float max3_abs(float m, float a, float b) {
  float r;
  asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
}

// spin_store<SpinH> with 32-bit offsets
__device__ __forceinline__ void quad_store(const FieldRef& f, uint32_t e, const cplx<float> v[12]) {
  float m = 0.f;
#pragma unroll
  for (int c = 0; c < 12; c++) m = max3_abs(m, v[c].re, v[c].im);
  const float inv = m >= 1.17549435e-38f ? 1.0f / m : 0.f;   // subnormal sites are stored as zero
  char* d = static_cast<char*>(f.data);
#pragma unroll
  for (int k = 0; k < 3; k++) {
    uint4 q;
    q.x = f2h(v[4 * k + 0].re * inv, v[4 * k + 0].im * inv);
    q.y = f2h(v[4 * k + 1].re * inv, v[4 * k + 1].im * inv);
    q.z = f2h(v[4 * k + 2].re * inv, v[4 * k + 2].im * inv);
    q.w = f2h(v[4 * k + 3].re * inv, v[4 * k + 3].im * inv);
    *reinterpret_cast<uint4*>(d + k * f.plane * 16 + (e << 4)) = q;
  }
  f.norm[e] = m;
}

__device__ __forceinline__ double norm2(const cplx<float> v[12]) {
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < 12; k++) {
    s = fma(double(v[k].re), double(v[k].re), s);
    s = fma(double(v[k].im), double(v[k].im), s);
  }
  return s;
}

template <int DAG, int KIND, int EPI>
__global__ void __launch_bounds__(256, CPSHIP_QUAD_WAVES) k_hop_quad(HopParams P) {
#pragma clang fp contract(off)   // every variant rounds the same way: the sums are written as fused multiply-adds
  const int Vcb = P.geom.Vcb, nb = P.nb;
  const int sb = (int)logical_block(blockIdx.x, gridDim.x, !(P.flags & HOP_NO_XCD_REMAP));
  int rhs, blk, b = 0;
  int64_t pslot = sb;
  if (P.flags & HOP_SPATIAL) {
    const int per_b = (int)gridDim.x >> 3;
    b = sb / per_b;
    const int n_in = sb - b * per_b;
    rhs = n_in / P.bpr_b;
    blk = n_in - rhs * P.bpr_b;
    pslot = (int64_t)rhs * (P.bpr_b << 3) + (int64_t)b * P.bpr_b + blk;
  } else {
    rhs = sb / P.bpr;
    blk = sb - rhs * P.bpr;
  }
  const uint32_t el = (uint32_t)blk * blockDim.x + threadIdx.x;
  const uint32_t q = P.nb_shift >= 0 ? el >> P.nb_shift : __umulhi(el, P.nb_magic) >> P.nb_mshift;
  const uint32_t j = el - q * (uint32_t)nb;
  const uint32_t site = (P.flags & HOP_SPATIAL) ? P.perm[(int64_t)b * P.perm_S + q] : q;
  uint32_t out_par, site_cb;
  if (KIND == KIND_DWF) {
    out_par = site >= (uint32_t)Vcb ? 1u : 0u;
    site_cb = site - out_par * (uint32_t)Vcb;
  } else {
    out_par = (uint32_t)P.out_parity;
    site_cb = site;
  }
  const uint32_t ns = out_par * (uint32_t)Vcb + site_cb;
  QuadSite Q;
  {
    const uint4 f = P.nbr[ns], g = P.nbr[2 * (int64_t)Vcb + ns];
    Q.idx[0] = f.x; Q.idx[1] = f.y; Q.idx[2] = f.z; Q.idx[3] = f.w;
    Q.idx[4] = g.x; Q.idx[5] = g.y; Q.idx[6] = g.z; Q.idx[7] = g.w;
  }
  const uint32_t per_rhs = (uint32_t)P.nsites_out * (uint32_t)nb;
  const uint32_t base = (uint32_t)rhs * per_rhs;   // first element of the rhs
  Q.stride = 16u * (uint32_t)nb;
  Q.e0 = (base + (KIND == KIND_DWF ? (1u - out_par) * (uint32_t)Vcb * (uint32_t)nb : 0u) + j) << 4;
  const uint32_t row = (threadIdx.x & 3) < 2 ? (threadIdx.x & 3) : 2u;
  Q.links = static_cast<const char*>(P.gauge.data) + (uint64_t)ns * 288 + row * 12;

  cplx<float> acc[12];
#pragma unroll
  for (int k = 0; k < 12; k++) acc[k] = cmk<float>(0.f, 0.f);
  constexpr int NA = CPSHIP_QUAD_AHEAD;
  QuadDir buf[8];
#define CPSHIP_QL(D) quad_load<D>(P, Q, buf[D]);
  // the loads of direction D + NA go out before the arithmetic of D
#define CPSHIP_QC(D)                                                                               \
  if constexpr ((D) + NA < 8) { quad_load<((D) + NA) & 7>(P, Q, buf[((D) + NA) & 7]); }            \
  __builtin_amdgcn_sched_barrier(0);                                                       \
  quad_compute<D, DAG>(buf[D], acc);                                                               \
  __builtin_amdgcn_sched_barrier(0);
  CPSHIP_QL(0)
  if constexpr (NA > 1) { CPSHIP_QL(1) }
  if constexpr (NA > 2) { CPSHIP_QL(2) }
  if constexpr (NA > 3) { CPSHIP_QL(3) }
  if constexpr (NA > 4) { CPSHIP_QL(4) }
  if constexpr (NA > 5) { CPSHIP_QL(5) }
  if constexpr (NA > 6) { CPSHIP_QL(6) }
  if constexpr (NA > 7) { CPSHIP_QL(7) }
  CPSHIP_QC(0) CPSHIP_QC(1) CPSHIP_QC(2) CPSHIP_QC(3) CPSHIP_QC(4) CPSHIP_QC(5) CPSHIP_QC(6) CPSHIP_QC(7)
#undef CPSHIP_QL
#undef CPSHIP_QC

  if constexpr (KIND == KIND_DWF) {
    // fifth dimension (as in hop_element): the slots s - 1, s + 1 of the
    // same 4-D site
    const int ls = P.ls;
    const int cls_out = (int)((out_par + (uint32_t)P.out_cb5) & 1u);
    const int s = 2 * (int)j + cls_out;
    const uint32_t site_base = base + ns * (uint32_t)nb;
    const int sm = (s == 0) ? ls - 1 : s - 1;
    const int sp = (s == ls - 1) ? 0 : s + 1;
    const float cw = float(P.neg_mass_two_over_a5), c2 = float(P.two_over_a5);
    const float cm = (s == 0) ? cw : c2, cp = (s == ls - 1) ? cw : c2;
    constexpr int c_from_m = (DAG == 0) ? 0 : 6, c_from_p = (DAG == 0) ? 6 : 0;
    uint32_t wm[6], wp[6];
    float nm, np;
    load_half_words(P.in, site_base + (uint32_t)(sm >> 1), c_from_m, wm, nm);
    load_half_words(P.in, site_base + (uint32_t)(sp >> 1), c_from_p, wp, np);
    const float fm = cm * nm, fp = cp * np;
#pragma unroll
    for (int k = 0; k < 6; k++) {
      fma_word(wm[k], fm, acc[c_from_m + k]);
      fma_word(wp[k], fp, acc[c_from_p + k]);
    }
  }

  const uint32_t eo = base + ns * (uint32_t)nb + j - (KIND == KIND_DWF ? 0u : out_par * (uint32_t)Vcb * (uint32_t)nb);
  cplx<float> res[12];
  if constexpr (EPI == QE_S5X || EPI == QE_S5XR || EPI == QE_S5XRR) {
    const int ls = nb, s = (int)j;
    const uint32_t sbase = eo - j;
    const float cm = (s == 0) ? -float(P.x5mass) : 1.f;
    const float cp = (s == ls - 1) ? -float(P.x5mass) : 1.f;
    constexpr int c_from_m = DAG ? 6 : 0, c_from_p = DAG ? 0 : 6;
    const float x5 = float(P.x5coef), sc = float(P.scale * P.hb5), xc = float(P.xcoef);
#pragma unroll
    for (int k = 0; k < 12; k++) res[k] = cmk<float>(sc * acc[k].re, sc * acc[k].im);
    // X and the s-term of X
    const int64_t pb = P.X.plane * 16;
    uint32_t xw[12];
    {
      uint4 t[3];
#pragma unroll
      for (int k = 0; k < 3; k++) t[k] = ld_off<uint4>(P.X.data, k * pb, eo << 4);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        xw[4 * k] = t[k].x; xw[4 * k + 1] = t[k].y; xw[4 * k + 2] = t[k].z; xw[4 * k + 3] = t[k].w;
      }
    }
    const float xn = ld_off<float>(P.X.norm, 0, eo << 2);
    uint32_t wm[6], wp[6];
    float nm, np;
    if constexpr (EPI == QE_S5X) {
      const int sm = (s == 0) ? ls - 1 : s - 1, sp = (s == ls - 1) ? 0 : s + 1;
      load_half_words(P.X, sbase + (uint32_t)sm, c_from_m, wm, nm);
      load_half_words(P.X, sbase + (uint32_t)sp, c_from_p, wp, np);
    } else {
      // the 16 slots of the site are one DPP row
#pragma unroll
      for (int k = 0; k < 6; k++) {
        wm[k] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)xw[c_from_m + k], DPP_ROW_ROR + 1, 0xF, 0xF, true);
        wp[k] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)xw[c_from_p + k], DPP_ROW_ROR + 15, 0xF, 0xF, true);
      }
      nm = dpp_f<DPP_ROW_ROR + 1>(xn);
      np = dpp_f<DPP_ROW_ROR + 15>(xn);
    }
    const float fx = xc * xn, fm = x5 * (cm * nm), fp = x5 * (cp * np);
#pragma unroll
    for (int k = 0; k < 12; k++) fma_word(xw[k], fx, res[k]);
#pragma unroll
    for (int k = 0; k < 6; k++) {
      fma_word(wm[k], fm, res[c_from_m + k]);
      fma_word(wp[k], fp, res[c_from_p + k]);
    }
    if (P.hc5 != 0.0) {
      // P applied to the hop itself: the hop of slots s - 1, s + 1 comes
      // from the neighbouring lanes of the site's aligned group
      const int lane = (int)(threadIdx.x & 63);
      const int lm = (s == 0) ? lane + ls - 1 : lane - 1;
      const int lp = (s == ls - 1) ? lane - (ls - 1) : lane + 1;
      const float scm = float(P.scale * P.hc5) * cm, scp = float(P.scale * P.hc5) * cp;
#pragma unroll
      for (int k = 0; k < 6; k++) {
        float mre, mim, pre, pim;
        if constexpr (EPI != QE_S5X) {
          mre = dpp_f<DPP_ROW_ROR + 1>(acc[c_from_m + k].re);
          mim = dpp_f<DPP_ROW_ROR + 1>(acc[c_from_m + k].im);
          pre = dpp_f<DPP_ROW_ROR + 15>(acc[c_from_p + k].re);
          pim = dpp_f<DPP_ROW_ROR + 15>(acc[c_from_p + k].im);
        } else {
          mre = __shfl(acc[c_from_m + k].re, lm, 64);
          mim = __shfl(acc[c_from_m + k].im, lm, 64);
          pre = __shfl(acc[c_from_p + k].re, lp, 64);
          pim = __shfl(acc[c_from_p + k].im, lp, 64);
        }
        res[c_from_m + k].re = fmaf(scm, mre, res[c_from_m + k].re);
        res[c_from_m + k].im = fmaf(scm, mim, res[c_from_m + k].im);
        res[c_from_p + k].re = fmaf(scp, pre, res[c_from_p + k].re);
        res[c_from_p + k].im = fmaf(scp, pim, res[c_from_p + k].im);
      }
    }
  } else {
    const float sc = float(P.scale);
#pragma unroll
    for (int k = 0; k < 12; k++) res[k] = cmk<float>(sc * acc[k].re, sc * acc[k].im);
    if constexpr (EPI == QE_X || EPI == QE_NRR) {
      const int64_t pb = P.X.plane * 16;
      uint4 t[3];
#pragma unroll
      for (int k = 0; k < 3; k++) t[k] = ld_off<uint4>(P.X.data, k * pb, eo << 4);
      const float fx = float(P.xcoef) * ld_off<float>(P.X.norm, 0, eo << 2);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        fma_word(t[k].x, fx, res[4 * k]);
        fma_word(t[k].y, fx, res[4 * k + 1]);
        fma_word(t[k].z, fx, res[4 * k + 2]);
        fma_word(t[k].w, fx, res[4 * k + 3]);
      }
    }
    if constexpr (EPI == QE_M5) m5_row<DAG>(P, (int)j, res);
  }

  if constexpr (EPI == QE_S5XRR || EPI == QE_NRR) {
    // the CG step r -= alpha (M^dag M p) and |r|^2, with M^dag M p in FP32
    double nrm = 0.0;
    if (P.ractive[rhs]) {
      const float a = float(P.ralpha[rhs]);
      const int64_t pb = P.R.plane * 16;
      uint4 t[3];
#pragma unroll
      for (int k = 0; k < 3; k++) t[k] = ld_off<uint4>(P.R.data, k * pb, eo << 4);
      const float rn = ld_off<float>(P.R.norm, 0, eo << 2);
#pragma unroll
      for (int k = 0; k < 12; k++) res[k] = cmk<float>(-a * res[k].re, -a * res[k].im);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        fma_word(t[k].x, rn, res[4 * k]);
        fma_word(t[k].y, rn, res[4 * k + 1]);
        fma_word(t[k].z, rn, res[4 * k + 2]);
        fma_word(t[k].w, rn, res[4 * k + 3]);
      }
      nrm = norm2(res);
      quad_store(P.R, eo, res);
    }
    if (P.partial) block_partial<double>(nrm, P.partial, pslot);
  } else {
    quad_store(P.out, eo, res);
    if (P.partial) block_partial<double>(norm2(res), P.partial, pslot);
  }
}

hipError_t launch_hop_quad(const HopParams& P, hipStream_t st) {
  const int bs = P.block;
  const int64_t per_rhs = (int64_t)P.nsites_out * P.nb;
  if (!quad_setup(P, bs) || !P.gauge.data) return hipErrorInvalidValue;
  // the reduction adds the partials of default blocks
  if (P.partial && bs != pick_block(per_rhs)) return hipErrorInvalidValue;
  HopParams Q = P;
  Q.bpr = (int)(per_rhs / bs);
  Q.bpr_b = (int)(((int64_t)P.perm_S * P.nb) / bs);
  if ((P.flags & HOP_SPATIAL) && (!P.perm || (int64_t)P.perm_S * P.nb % bs || Q.bpr_b < 1 ||
                                  (int64_t)Q.bpr_b * 8 != Q.bpr || (P.flags & HOP_NO_XCD_REMAP)))
    return hipErrorInvalidValue;
  Q.nb_shift = (P.nb & (P.nb - 1)) == 0 ? __builtin_ctz((unsigned)P.nb) : -1;
  // division by nb of dividends below 2^31: (el * magic) >> (32 + mshift)
  // with magic = ceil(2^(32 + mshift) / nb), mshift = ceil(log2 nb) - 1
  Q.nb_mshift = 31 - __builtin_clz((unsigned)P.nb - 1);
  Q.nb_magic = (uint32_t)(((uint64_t(1) << (32 + Q.nb_mshift)) + P.nb - 1) / P.nb);
  const dim3 grid((unsigned)((int64_t)Q.bpr * P.nrhs)), block(bs);
  const bool dwf = P.kind == KIND_DWF;
#define CPSHIP_QUAD(KIND, EPI)                                                                   \
  {                                                                                              \
    if (P.dag) hipLaunchKernelGGL((k_hop_quad<1, KIND, EPI>), grid, block, 0, st, Q);            \
    else hipLaunchKernelGGL((k_hop_quad<0, KIND, EPI>), grid, block, 0, st, Q);                  \
    return hipGetLastError();                                                                    \
  }
  if (P.rupd && (!P.R.data || !P.R.norm || !P.ralpha || !P.ractive)) return hipErrorInvalidValue;
  if (P.clov == CLOV_NONE && !P.rupd && !P.m5post) {
    if (P.X.data) {
      if (dwf) CPSHIP_QUAD(KIND_DWF, QE_X) else CPSHIP_QUAD(KIND_WILSON, QE_X)
    }
    if (dwf) CPSHIP_QUAD(KIND_DWF, QE_PLAIN) else CPSHIP_QUAD(KIND_WILSON, QE_PLAIN)
  }
  if (P.clov == CLOV_NONE && P.m5post) {
    if (dwf || P.rupd || P.nb != 16 || P.X.data) return hipErrorInvalidValue;
    CPSHIP_QUAD(KIND_WILSON, QE_M5)
  }
  if (P.clov == CLOV_NONE) {
    if (!dwf || !P.X.data) return hipErrorInvalidValue;
    CPSHIP_QUAD(KIND_DWF, QE_NRR)
  }
  if (P.clov != CLOV_S5X || dwf || !P.X.data || P.m5post) return hipErrorInvalidValue;
  // the fused P hop term reads slots s-1, s+1 from lanes of one wavefront
  if (P.hc5 != 0.0 && 64 % P.nb) return hipErrorInvalidValue;
  if (P.s5_row && P.nb != 16) return hipErrorInvalidValue;
  if (P.rupd) {
    if (!P.s5_row) return hipErrorInvalidValue;
    CPSHIP_QUAD(KIND_WILSON, QE_S5XRR)
  }
  if (P.s5_row) CPSHIP_QUAD(KIND_WILSON, QE_S5XR)
  CPSHIP_QUAD(KIND_WILSON, QE_S5X)
#undef CPSHIP_QUAD
}

// Links of the quad hop: for every (parity, site) the links of directions
// d = 0..7 onto it, 9 words (FP16 pairs) each, row major: U_mu(x) forward and
// U_mu(x - mu)^dagger backward, an element u as (re u, -im u).
// BF16 storage keeps BF16-rounded numbers, as the FP16 the product uses.
template <bool BF16>
__global__ void __launch_bounds__(256) k_pack_gauge_quad(const double* __restrict__ aos, uint32_t* __restrict__ out,
                                                         const uint4* __restrict__ nbr, int Vcb) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)16 * Vcb) return;
  const int d = (int)(t & 7), mu = d & 3;
  const int64_t ns = t >> 3;
  const int par = ns >= Vcb ? 1 : 0;
  int64_t src = ns;
  if (d >= 4) {
    const uint32_t n = reinterpret_cast<const uint32_t*>(nbr)[(2 * (int64_t)Vcb + ns) * 4 + mu];
    src = (int64_t)(1 - par) * Vcb + n;
  }
  const double* u = aos + 72 * src + 18 * mu;
  uint32_t* o = out + 9 * t;
  for (int r = 0; r < 3; r++)
    for (int c = 0; c < 3; c++) {
      // WILSON order holds U(row, col) at 2 (row + 3 col)
      const int k = d < 4 ? 2 * (r + 3 * c) : 2 * (c + 3 * r);
      float re = float(u[k]), im = float(u[k + 1]);
      if (BF16) {
        re = __bfloat162float(__float2bfloat16(re));
        im = __bfloat162float(__float2bfloat16(im));
      }
      // row r of U or U^dagger, elements as (re, -im)
      o[3 * r + c] = f2h(re, d < 4 ? -im : im);
    }
}

hipError_t pack_gauge_quad(bool bf16, const double* aos, void* out, const uint4* nbr, int Vcb, hipStream_t st) {
  const dim3 grid((unsigned)(((int64_t)16 * Vcb + 255) / 256)), block(256);
  uint32_t* o = static_cast<uint32_t*>(out);
  if (bf16) hipLaunchKernelGGL(k_pack_gauge_quad<true>, grid, block, 0, st, aos, o, nbr, Vcb);
  else hipLaunchKernelGGL(k_pack_gauge_quad<false>, grid, block, 0, st, aos, o, nbr, Vcb);
  return hipGetLastError();
}

}  // namespace cpship
