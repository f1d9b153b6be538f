// Device building blocks of the hopping term: spin projection, SU(3) x
// half-spinor, reconstruction.  Operator and leg order as the reference Hand
// kernel (WilsonKernelsHandCpu.h:426-446): leg d reads the neighbour in
// direction d (Xp Yp Zp Tp Xm Ym Zm Tm) and link U[x][d]; non-dagger uses the
// projector *M_PROJ on forward legs and *P_PROJ on backward legs
// (WilsonKernelsHandCpu.h:94-159, 165-303); the dagger swaps them.
#pragma once

#include "layout_dev.h"

namespace dev {

enum { PXP = 0, PYP, PZP, PTP, PXM, PYM, PZM, PTM };

__device__ __forceinline__ float dfma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double dfma(double a, double b, double c) { return __builtin_fma(a, b, c); }

// Projector kind used on leg `dir`.
template <bool DAG, int DIR> struct LegProj {
  static constexpr int value = DAG ? DIR : (DIR ^ 4);
};

// Sums and differences of a neighbour spinor's reals, real 2*(sp*3+c) + {0,1}
// = re/im of spin sp colour c: of an array in the arithmetic type, ...
template <typename A> struct Reals {
  const A *v;
  __device__ __forceinline__ A add(int i, int j) const { return v[i] + v[j]; }
  __device__ __forceinline__ A sub(int i, int j) const { return v[i] - v[j]; }
};

// ... or of 16-bit chunks as they were loaded.  FP16: one v_fma_mix_f32 (a * 1
// + b with both read as halves of a register), which takes the place of two
// conversions and an addition; `one` is 1.0f the compiler cannot fold.  Both
// round the exact sum once.
template <int P> struct RawReals {
  typename Traits<P>::vec c[Traits<P>::NCH];
  float one;
  __device__ __forceinline__ float real(int i) const { return (float)c[i >> 3][i & 7]; }
  __device__ __forceinline__ float add(int i, int j) const
  {
    if constexpr (P == GBX_F16) return __builtin_fmaf(real(i), one, real(j));
    else return real(i) + real(j);
  }
  __device__ __forceinline__ float sub(int i, int j) const
  {
    if constexpr (P == GBX_F16) return __builtin_fmaf(real(i), one, -real(j));
    else return real(i) - real(j);
  }
};

// h[0..2] = upper half-spinor row 0, h[3..5] = row 1 (re in hr, im in hi).
template <int K, typename V, typename A>
__device__ __forceinline__ void project_from(const V &v, A *hr, A *hi)
{
#define PR(sp, c) (2 * ((sp) * 3 + (c)))
#define PI(sp, c) (2 * ((sp) * 3 + (c)) + 1)
#pragma unroll
  for (int c = 0; c < 3; c++) {
    if (K == PXP) {  // h0 = p0 + i p3, h1 = p1 + i p2
      hr[c] = v.sub(PR(0, c), PI(3, c)); hi[c] = v.add(PI(0, c), PR(3, c));
      hr[3 + c] = v.sub(PR(1, c), PI(2, c)); hi[3 + c] = v.add(PI(1, c), PR(2, c));
    } else if (K == PYP) {  // h0 = p0 - p3, h1 = p1 + p2
      hr[c] = v.sub(PR(0, c), PR(3, c)); hi[c] = v.sub(PI(0, c), PI(3, c));
      hr[3 + c] = v.add(PR(1, c), PR(2, c)); hi[3 + c] = v.add(PI(1, c), PI(2, c));
    } else if (K == PZP) {  // h0 = p0 + i p2, h1 = p1 - i p3
      hr[c] = v.sub(PR(0, c), PI(2, c)); hi[c] = v.add(PI(0, c), PR(2, c));
      hr[3 + c] = v.add(PR(1, c), PI(3, c)); hi[3 + c] = v.sub(PI(1, c), PR(3, c));
    } else if (K == PTP) {  // h0 = p0 + p2, h1 = p1 + p3
      hr[c] = v.add(PR(0, c), PR(2, c)); hi[c] = v.add(PI(0, c), PI(2, c));
      hr[3 + c] = v.add(PR(1, c), PR(3, c)); hi[3 + c] = v.add(PI(1, c), PI(3, c));
    } else if (K == PXM) {  // h0 = p0 - i p3, h1 = p1 - i p2
      hr[c] = v.add(PR(0, c), PI(3, c)); hi[c] = v.sub(PI(0, c), PR(3, c));
      hr[3 + c] = v.add(PR(1, c), PI(2, c)); hi[3 + c] = v.sub(PI(1, c), PR(2, c));
    } else if (K == PYM) {  // h0 = p0 + p3, h1 = p1 - p2
      hr[c] = v.add(PR(0, c), PR(3, c)); hi[c] = v.add(PI(0, c), PI(3, c));
      hr[3 + c] = v.sub(PR(1, c), PR(2, c)); hi[3 + c] = v.sub(PI(1, c), PI(2, c));
    } else if (K == PZM) {  // h0 = p0 - i p2, h1 = p1 + i p3
      hr[c] = v.add(PR(0, c), PI(2, c)); hi[c] = v.sub(PI(0, c), PR(2, c));
      hr[3 + c] = v.sub(PR(1, c), PI(3, c)); hi[3 + c] = v.add(PI(1, c), PR(3, c));
    } else {  // PTM: h0 = p0 - p2, h1 = p1 - p3
      hr[c] = v.sub(PR(0, c), PR(2, c)); hi[c] = v.sub(PI(0, c), PI(2, c));
      hr[3 + c] = v.sub(PR(1, c), PR(3, c)); hi[3 + c] = v.sub(PI(1, c), PI(3, c));
    }
  }
#undef PR
#undef PI
}

template <int K, typename A>
__device__ __forceinline__ void project(const A *v, A *hr, A *hi)
{
  project_from<K>(Reals<A>{v}, hr, hi);
}

// The reference's arithmetic for U x chi: every complex product
// (ar*br - ai*bi, ar*bi + ai*br) rounded term by term, summed over the
// columns left to right, t = U_i0 chi_0; t += U_i1 chi_1; t += U_i2 chi_2
// (WilsonKernelsHandCpu.h:62-90, arch/generic/Simd_generic.h:153-155).
// No multiply-add is fused, so the result is the reference's to the bit.
template <typename A>
__device__ __forceinline__ void su3_mul_exact(const A *U, const A *hr, const A *hi, A *ur, A *ui)
{
#pragma clang fp contract(off)
#pragma unroll
  for (int sp = 0; sp < 2; sp++)
#pragma unroll
    for (int i = 0; i < 3; i++) {
      A re = U[(i * 3) * 2] * hr[sp * 3] - U[(i * 3) * 2 + 1] * hi[sp * 3];
      A im = U[(i * 3) * 2] * hi[sp * 3] + U[(i * 3) * 2 + 1] * hr[sp * 3];
#pragma unroll
      for (int j = 1; j < 3; j++) {
        const A pr = U[(i * 3 + j) * 2] * hr[sp * 3 + j] - U[(i * 3 + j) * 2 + 1] * hi[sp * 3 + j];
        const A pi = U[(i * 3 + j) * 2] * hi[sp * 3 + j] + U[(i * 3 + j) * 2 + 1] * hr[sp * 3 + j];
        re = re + pr;
        im = im + pi;
      }
      ur[sp * 3 + i] = re;
      ui[sp * 3 + i] = im;
    }
}

// u[sp*3+i] = sum_j U[i][j] h[sp*3+j]; U row-major complex, 18 reals.
// MUL_CHAIN: one multiply + five fused multiply-adds per real output (72 ops
// per leg, 840 VALU ops per 5D site instead of 1032 for the mul/fma/add form
// the compiler derives from the plain expression).  MUL_EXACT: the
// reference's rounding.
enum { MUL_CHAIN = 0, MUL_EXACT = 1 };
template <int MUL, typename A>
__device__ __forceinline__ void su3_mul(const A *U, const A *hr, const A *hi, A *ur, A *ui)
{
  if constexpr (MUL == MUL_EXACT) {
    su3_mul_exact(U, hr, hi, ur, ui);
    return;
  }
#pragma unroll
  for (int sp = 0; sp < 2; sp++)
#pragma unroll
    for (int i = 0; i < 3; i++) {
      A re = U[(i * 3) * 2] * hr[sp * 3];
      A im = U[(i * 3) * 2] * hi[sp * 3];
      re = dfma(-U[(i * 3) * 2 + 1], hi[sp * 3], re);
      im = dfma(U[(i * 3) * 2 + 1], hr[sp * 3], im);
#pragma unroll
      for (int j = 1; j < 3; j++) {
        re = dfma(U[(i * 3 + j) * 2], hr[sp * 3 + j], re);
        im = dfma(U[(i * 3 + j) * 2], hi[sp * 3 + j], im);
        re = dfma(-U[(i * 3 + j) * 2 + 1], hi[sp * 3 + j], re);
        im = dfma(U[(i * 3 + j) * 2 + 1], hr[sp * 3 + j], im);
      }
      ur[sp * 3 + i] = re;
      ui[sp * 3 + i] = im;
    }
}

// Accumulate (FIRST: assign) the reconstructed 4-spinor of kind K.
// u0 = (ur[0..2], ui[0..2]), u1 = (ur[3..5], ui[3..5]); r index sp*3+c.
template <int K, bool FIRST, typename A>
__device__ __forceinline__ void recon(const A *ur, const A *ui, A *rr, A *ri)
{
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const A u0r = ur[c], u0i = ui[c], u1r = ur[3 + c], u1i = ui[3 + c];
    if (FIRST) {
      rr[c] = u0r; ri[c] = u0i;
      rr[3 + c] = u1r; ri[3 + c] = u1i;
      if (K == PXP) {  // r2 = -i u1, r3 = -i u0
        rr[6 + c] = u1i; ri[6 + c] = -u1r;
        rr[9 + c] = u0i; ri[9 + c] = -u0r;
      } else {  // PXM: r2 = i u1, r3 = i u0
        rr[6 + c] = -u1i; ri[6 + c] = u1r;
        rr[9 + c] = -u0i; ri[9 + c] = u0r;
      }
      continue;
    }
    rr[c] += u0r; ri[c] += u0i;
    rr[3 + c] += u1r; ri[3 + c] += u1i;
    if (K == PXP) {  // r2 -= i u1, r3 -= i u0
      rr[6 + c] += u1i; ri[6 + c] -= u1r;
      rr[9 + c] += u0i; ri[9 + c] -= u0r;
    } else if (K == PXM) {  // r2 += i u1, r3 += i u0
      rr[6 + c] -= u1i; ri[6 + c] += u1r;
      rr[9 + c] -= u0i; ri[9 + c] += u0r;
    } else if (K == PYP) {  // r2 += u1, r3 -= u0
      rr[6 + c] += u1r; ri[6 + c] += u1i;
      rr[9 + c] -= u0r; ri[9 + c] -= u0i;
    } else if (K == PYM) {  // r2 -= u1, r3 += u0
      rr[6 + c] -= u1r; ri[6 + c] -= u1i;
      rr[9 + c] += u0r; ri[9 + c] += u0i;
    } else if (K == PZP) {  // r2 -= i u0, r3 += i u1
      rr[6 + c] += u0i; ri[6 + c] -= u0r;
      rr[9 + c] -= u1i; ri[9 + c] += u1r;
    } else if (K == PZM) {  // r2 += i u0, r3 -= i u1
      rr[6 + c] -= u0i; ri[6 + c] += u0r;
      rr[9 + c] += u1i; ri[9 + c] -= u1r;
    } else if (K == PTP) {  // r2 += u0, r3 += u1
      rr[6 + c] += u0r; ri[6 + c] += u0i;
      rr[9 + c] += u1r; ri[9 + c] += u1i;
    } else {  // PTM: r2 -= u0, r3 -= u1
      rr[6 + c] -= u0r; ri[6 + c] -= u0i;
      rr[9 + c] -= u1r; ri[9 + c] -= u1i;
    }
  }
}

// Third row of an SU(3) matrix from the first two: row2 = conj(row0 x row1).
template <typename A>
__device__ __forceinline__ void su3_row2(A *U)
{
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const int a = (j + 1) % 3, b = (j + 2) % 3;
    const A ar = U[a * 2], ai = U[a * 2 + 1], br = U[6 + b * 2], bi = U[6 + b * 2 + 1];
    const A cr = U[b * 2], ci = U[b * 2 + 1], dr = U[6 + a * 2], di = U[6 + a * 2 + 1];
    const A xr = (ar * br - ai * bi) - (cr * dr - ci * di);
    const A xi = (ar * bi + ai * br) - (cr * di + ci * dr);
    U[12 + j * 2] = xr;
    U[12 + j * 2 + 1] = -xi;
  }
}

// Stage the links (and neighbour slots) of workgroup sites q0 .. q0+nsl-1
// into LDS as accumulation-precision 3x3 matrices [site][dir][18].
// A workgroup can gather nothing before this is done, so it should cost one
// memory round trip: the neighbour slots and up to N 16-byte pieces of links a
// thread are all loaded before the first is stored to LDS (N covers a default
// shape with minor extents from 6 on).  One real at a time, each waited for, it
// was 9 round trips in FP64 at Ls 16 and 18 at Ls 8: FP64 8^4 x Ls8 6.8 -> 4.8
// us; FP32 20x18x10x14 x Ls10 37.2 -> 36.0 us; FP64 24^4 x Ls16 747 -> 735 us;
// CG at 16^3x24 x Ls8, FP16 inner, 11.7 -> 9.6 ms, domain-wall solve 16^4 x
// Ls12, FP32 inner, 15.2 -> 13.5 ms.  With many right-hand sides, where a
// workgroup's staging was short before, it is level or 1 % behind (FP32 16^4 x
// Ls16 x 8: 597 -> 605 us).
template <int P, bool C12>
__device__ __forceinline__ void stage_links(const void *__restrict__ gauge, const uint32_t *__restrict__ nbr, uint32_t q0,
                                            uint32_t nsl, typename Traits<P>::acc *sU, uint32_t *sN, uint32_t scale = 1)
{
  typedef typename Traits<P>::acc A;
  typedef typename Traits<P>::st S;
  typedef typename Traits<P>::vec V;
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  constexpr int RL = C12 ? 12 : 18, R = Traits<P>::R, PS = 8 * RL / R;  // pieces of a site
  constexpr int N = P == GBX_F64 ? 12 : P == GBX_F32 ? 8 : 4;
  const V *g = (const V *)((const S *)gauge + (uint64_t)q0 * 8 * RL);
  const u4 *gn = (const u4 *)(nbr + (uint64_t)q0 * 8);
  const uint32_t n = nsl * PS, nn = nsl * 2, th = blockDim.x;
  u4 nb;
  if (threadIdx.x < nn) nb = gn[threadIdx.x];
  for (uint32_t e0 = threadIdx.x; e0 < n; e0 += N * th) {
    V x[N];
    // Links are read once per launch: non-temporal loads keep them from
    // displacing neighbour spinors, which are re-read, in the L2.
#pragma unroll
    for (int i = 0; i < N; i++)
      if (e0 + i * th < n) x[i] = __builtin_nontemporal_load(g + e0 + i * th);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < N; i++) {
      const uint32_t e = e0 + i * th;
      if (e >= n) break;
      if constexpr (!C12 && R * sizeof(A) == 16) {
        ((V *)sU)[e] = x[i];
      } else {
#pragma unroll
        for (int j = 0; j < R; j += 2) {  // a link's reals are even in number
          const uint32_t r = e * R + j, link = r / RL;
          A *d = sU + link * (18 - RL) + r;
          d[0] = (A)x[i][j];
          d[1] = (A)x[i][j + 1];
        }
      }
    }
  }
  for (uint32_t e = threadIdx.x; e < nn; e += th) {
    if (e != threadIdx.x) nb = gn[e];
    ((u4 *)sN)[e] = nb * scale;
  }
  if (C12) {
    __syncthreads();
    for (uint32_t l = threadIdx.x; l < nsl * 8; l += blockDim.x) su3_row2(sU + l * 18);
  }
  __syncthreads();
}

// Chunk k of neighbour `nb`, minor index m: `nb` is its slot, or for O32 its byte
// offset in a field of at most 4 GiB.  The chunk's address is then a scalar base
// (the field's, k chunks on) and a 32-bit offset, one addition a leg in place of
// a 64-bit multiplication and an addition a load: about 100 of a point's 1000
// VALU operations and a few registers.  The solvers' FP32 and 16-bit forms take
// it (their hops read from the caches, where the arithmetic shows): CG at
// 16^3x24 x Ls8, FP16 inner, 11.72 -> 11.33 ms, domain-wall solve 16^4 x Ls12,
// FP32 inner, 15.08 -> 14.76 ms.  The others are bound by the L2 misses and run
// no faster or up to 1.6 % slower (24^4 x Ls16 FP64 748 -> 760 us; BF16 16^3x24
// x Ls12 x 16 704 either way), as their gathers then come in denser bursts.
template <int P, bool O32>
__device__ __forceinline__ typename Traits<P>::vec load_at(const void *__restrict__ in, uint32_t nb, uint32_t M, uint32_t m, int k)
{
  typedef typename Traits<P>::vec V;
  if constexpr (O32) {
    typedef const __attribute__((address_space(1))) char *G;
    G base = (G)in + (uint64_t)k * M * 16;
    asm("" : "+s"(base));  // kept apart from the offset
    return *(const __attribute__((address_space(1))) V *)(base + (nb + m * 16));
  } else {
    return ((const V *)in)[(uint64_t)nb * Traits<P>::NCH * M + m + (uint64_t)k * M];
  }
}

// Gather the 24 reals of a neighbour.
template <int P, bool O32 = false>
__device__ __forceinline__ void load_nb(const void *__restrict__ in, uint32_t nb, uint32_t M, uint32_t m,
                                        typename Traits<P>::acc *v)
{
  constexpr int NCH = Traits<P>::NCH, R = Traits<P>::R;
#pragma unroll
  for (int k = 0; k < NCH; k++) {
    const typename Traits<P>::vec x = load_at<P, O32>(in, nb, M, m, k);
#pragma unroll
    for (int j = 0; j < R; j++) v[k * R + j] = (typename Traits<P>::acc)x[j];
  }
}

// project, multiply by U (18 reals in LDS), reconstruct into r
template <int K, bool FIRST, int MUL, typename A>
__device__ __forceinline__ void leg_compute(const A *v, const A *U, A *rr, A *ri)
{
  A hr[6], hi[6], ur[6], ui[6];
  project<K>(v, hr, hi);
  su3_mul<MUL>(U, hr, hi, ur, ui);
  recon<K, FIRST>(ur, ui, rr, ri);
}

// Legs of a domain part whose ghosts hold projected halves.  Neighbour slot
// n >= ghost0 is half-slot n - ghost0 of the ghost region (NCH/2 chunks per
// half-slot, after the ghost0 whole slots): its chunks k and k + NCH/2 are
// both read from half-slot chunk k (the same lines, so the second read hits
// the cache), v[0..11] then holds the two-spinor, and the leg uses it in
// place of its projection.  Other neighbours are gathered and projected as
// in dhop_site; the arithmetic is the same.
template <int P>
__device__ __forceinline__ bool load_nb_gp(const void *__restrict__ in, uint32_t nb, uint32_t M, uint32_t m,
                                           uint32_t ghost0, typename Traits<P>::acc *v)
{
  constexpr int NCH = Traits<P>::NCH, HCH = NCH / 2, R = Traits<P>::R;
  const bool g = nb >= ghost0;
  const uint64_t full = (uint64_t)nb * NCH * M + m;
  const uint64_t half = (uint64_t)ghost0 * NCH * M + (uint64_t)(g ? nb - ghost0 : 0) * HCH * M + m;
#pragma unroll
  for (int k = 0; k < NCH; k++) {
    const uint64_t t = g ? half + (uint64_t)(k % HCH) * M : full + (uint64_t)k * M;
    load_chunk<P, typename Traits<P>::acc>(in, t, v + k * R);
  }
  return g;
}

template <int K, bool FIRST, int MUL, typename A>
__device__ __forceinline__ void leg_compute_gp(const A *v, bool g, const A *U, A *rr, A *ri)
{
  A hr[6], hi[6], ur[6], ui[6];
  project<K>(v, hr, hi);
#pragma unroll
  for (int j = 0; j < 6; j++) {
    hr[j] = g ? v[2 * j] : hr[j];
    hi[j] = g ? v[2 * j + 1] : hi[j];
  }
  su3_mul<MUL>(U, hr, hi, ur, ui);
  recon<K, FIRST>(ur, ui, rr, ri);
}

// GBX_BASIS_TDIAG fields (psi' = S psi, S = [[1, 1], [1, -1]] / sqrt(2) on
// the spin pairs (0, 2), (1, 3)): there gamma_x,y,z are the chiral ones
// negated, so an x, y or z leg uses the projector kind of the opposite sign,
// and gamma_t = diag(1, 1, -1, -1), so the t legs' projectors 1 +/- gamma_t
// keep twice the upper (kind PTP) or lower (PTM) two spins: such a leg
// gathers NCH/2 chunks, multiplies them by the link and adds twice the
// product to that half of the result.
template <bool DAG, int D, bool TD> struct LegKind {
  static constexpr int value = LegProj<DAG, D>::value ^ ((TD && (D & 3) != 3) ? 4 : 0);
};
template <bool DAG, int D, bool TD> struct LegHalf {
  static constexpr bool value = TD && (D & 3) == 3;              // gathers half a spinor
  static constexpr bool upper = LegProj<DAG, D>::value == PTP;  // which half
};

// Chunks of one spin half (v[0..11] = its 2 spins x 3 colours).
template <int P, bool UPPER, bool O32 = false>
__device__ __forceinline__ void load_nb_half(const void *__restrict__ in, uint32_t nb, uint32_t M, uint32_t m,
                                             typename Traits<P>::acc *v)
{
  constexpr int NCH = Traits<P>::NCH, R = Traits<P>::R, K0 = UPPER ? 0 : NCH / 2;
#pragma unroll
  for (int k = 0; k < NCH / 2; k++) {
    const typename Traits<P>::vec x = load_at<P, O32>(in, nb, M, m, K0 + k);
#pragma unroll
    for (int j = 0; j < R; j++) v[k * R + j] = (typename Traits<P>::acc)x[j];
  }
}

template <bool UPPER, int MUL, typename A>
__device__ __forceinline__ void leg_half(const A *v, const A *U, A *rr, A *ri)
{
  A hr[6], hi[6], ur[6], ui[6];
#pragma unroll
  for (int j = 0; j < 6; j++) {
    hr[j] = v[2 * j];
    hi[j] = v[2 * j + 1];
  }
  su3_mul<MUL>(U, hr, hi, ur, ui);
  constexpr int o = UPPER ? 0 : 6;
#pragma unroll
  for (int j = 0; j < 6; j++) {
    rr[o + j] = dfma((A)2, ur[j], rr[o + j]);
    ri[o + j] = dfma((A)2, ui[j], ri[o + j]);
  }
}

template <int P, bool DAG, int D, bool TD, bool O32 = false>
__device__ __forceinline__ void leg_load(const void *__restrict__ in, uint32_t nb, uint32_t M, uint32_t m,
                                         typename Traits<P>::acc *v)
{
  if constexpr (LegHalf<DAG, D, TD>::value) load_nb_half<P, LegHalf<DAG, D, TD>::upper, O32>(in, nb, M, m, v);
  else load_nb<P, O32>(in, nb, M, m, v);
}

// The leg arithmetic runs at raised wave priority (s_setprio 1), the gathers
// at the normal one: a wavefront holding a gathered leg finishes it and
// issues its next gathers sooner, which evens out the stream of gathers
// (FP64: about 1 % on TDIAG fields, 1.7 % on chiral fields; the arithmetic
// and its results are unchanged).
template <bool DAG, int D, bool TD, bool FIRST, int MUL, typename A>
__device__ __forceinline__ void leg_apply(const A *v, const A *U, A *rr, A *ri)
{
  static_assert(!(FIRST && LegHalf<DAG, D, TD>::value), "a half leg never comes first");
  __builtin_amdgcn_s_setprio(1);
  if constexpr (LegHalf<DAG, D, TD>::value) leg_half<LegHalf<DAG, D, TD>::upper, MUL>(v, U, rr, ri);
  else leg_compute<LegKind<DAG, D, TD>::value, FIRST, MUL>(v, U, rr, ri);
  __builtin_amdgcn_s_setprio(0);
}

// An empty asm that reads and redefines the accumulators: every leg's
// arithmetic is complete before the next leg's loads (otherwise the compiler
// sinks all legs' arithmetic below all loads and keeps eight gathered
// spinors live).
template <typename A>
__device__ __forceinline__ void pin_acc(A *rr, A *ri)
{
  asm volatile("" : "+v"(rr[0]), "+v"(rr[1]), "+v"(rr[2]), "+v"(rr[3]), "+v"(rr[4]), "+v"(rr[5]), "+v"(rr[6]),
               "+v"(rr[7]), "+v"(rr[8]), "+v"(rr[9]), "+v"(rr[10]), "+v"(rr[11]));
  asm volatile("" : "+v"(ri[0]), "+v"(ri[1]), "+v"(ri[2]), "+v"(ri[3]), "+v"(ri[4]), "+v"(ri[5]), "+v"(ri[6]),
               "+v"(ri[7]), "+v"(ri[8]), "+v"(ri[9]), "+v"(ri[10]), "+v"(ri[11]));
}

// 16-bit storage: the legs work on the chunks as loaded (12 registers a leg
// instead of 24), converted by the projection.  What bounds these kernels is
// the VALU as much as the gathers: 24^4 x Ls16 FP16, converting on load and with
// unchained products, took 1250 operations a point (190 of 243 us); 880 here,
// 211 us.  BF16 keeps its conversions: 1075.  16^3x24 x Ls12 x 16 BF16: 777 ->
// 659 us.
template <int P, bool O32 = false>
__device__ __forceinline__ void load_raw(const void *__restrict__ in, uint32_t nb, uint32_t M, uint32_t m, RawReals<P> &v)
{
#pragma unroll
  for (int k = 0; k < Traits<P>::NCH; k++) v.c[k] = load_at<P, O32>(in, nb, M, m, k);
}

template <int P, bool DAG, int D>
__device__ __forceinline__ void leg_raw(const RawReals<P> &v, const float *U, float *rr, float *ri)
{
  float hr[6], hi[6], ur[6], ui[6];
  __builtin_amdgcn_s_setprio(1);
  project_from<LegProj<DAG, D>::value>(v, hr, hi);
  su3_mul<MUL_CHAIN>(U, hr, hi, ur, ui);
  recon<LegProj<DAG, D>::value, D == 0>(ur, ui, rr, ri);
  __builtin_amdgcn_s_setprio(0);
}

// PF legs are gathered ahead of the one being computed; the scheduling barrier
// and the pinned accumulators keep the compiler from gathering (and holding)
// more of them, or from sinking the arithmetic into the stores' branches.
template <int P, bool DAG, int PF, bool O32>
__device__ __forceinline__ void dhop_site_raw(const void *__restrict__ in, const uint32_t *nb, uint32_t M, uint32_t m,
                                              const float *U, float *rr, float *ri)
{
  float one = 1.0f;
  if (P == GBX_F16) asm volatile("" : "+s"(one));
  RawReals<P> v[PF + 1];
#pragma unroll
  for (int d = 0; d <= PF; d++) v[d].one = one;
#pragma unroll
  for (int d = 0; d < PF; d++) load_raw<P, O32>(in, nb[d], M, m, v[d]);
#define GBX_RLEG(D)                                                                \
  if (D + PF < 8) load_raw<P, O32>(in, nb[(D + PF) & 7], M, m, v[(D + PF) % (PF + 1)]); \
  __builtin_amdgcn_sched_barrier(0);                                               \
  leg_raw<P, DAG, D>(v[D % (PF + 1)], U + D * 18, rr, ri);                         \
  pin_acc(rr, ri);                                                                 \
  __builtin_amdgcn_sched_barrier(0);
  GBX_RLEG(0)
  GBX_RLEG(1)
  GBX_RLEG(2)
  GBX_RLEG(3)
  GBX_RLEG(4)
  GBX_RLEG(5)
  GBX_RLEG(6)
  GBX_RLEG(7)
#undef GBX_RLEG
}

// Full 8-leg hopping term for (site with links U, neighbours nb[8], minor m).
// PF = 0: gather and compute leg by leg.  PF = 1: the gather of leg d+1 is
// issued before leg d is computed (two gather buffers in registers), which
// keeps a second set of loads in flight per wavefront.  PF = 2: three
// buffers, gathers two legs ahead.  EXACT: the reference's rounding in the
// SU(3) products (FP64 / FP32).  TD: GBX_BASIS_TDIAG fields (LegKind, LegHalf).
template <int P, bool DAG, int PF, bool EXACT = false, bool TD = false, bool O32 = false>
__device__ __forceinline__ void dhop_site(const void *__restrict__ in, const uint32_t *nb, uint32_t M, uint32_t m,
                                          const typename Traits<P>::acc *U, typename Traits<P>::acc *rr,
                                          typename Traits<P>::acc *ri)
{
  typedef typename Traits<P>::acc A;
  constexpr int CH = EXACT ? MUL_EXACT : MUL_CHAIN;
  if constexpr (P == GBX_F16 || P == GBX_BF16) {
    static_assert(!EXACT && !TD, "FP64 / FP32 forms");
    dhop_site_raw<P, DAG, PF, O32>(in, nb, M, m, U, rr, ri);
  } else if (PF == 0) {
    A v[24];
#define GBX_LEG(D, FIRST)                                                  \
    leg_load<P, DAG, D, TD, O32>(in, nb[D], M, m, v);                           \
    leg_apply<DAG, D, TD, FIRST, CH>(v, U + D * 18, rr, ri);
    GBX_LEG(0, true)
    GBX_LEG(1, false)
    GBX_LEG(2, false)
    GBX_LEG(3, false)
    GBX_LEG(4, false)
    GBX_LEG(5, false)
    GBX_LEG(6, false)
    GBX_LEG(7, false)
#undef GBX_LEG
  } else if (PF == 2) {
    A v0[24], v1[24], v2[24];
    leg_load<P, DAG, 0, TD, O32>(in, nb[0], M, m, v0);
    leg_load<P, DAG, 1, TD, O32>(in, nb[1], M, m, v1);
    leg_load<P, DAG, 2, TD, O32>(in, nb[2], M, m, v2);
    leg_apply<DAG, 0, TD, true, CH>(v0, U + 0 * 18, rr, ri);
    leg_load<P, DAG, 3, TD, O32>(in, nb[3], M, m, v0);
    leg_apply<DAG, 1, TD, false, CH>(v1, U + 1 * 18, rr, ri);
    leg_load<P, DAG, 4, TD, O32>(in, nb[4], M, m, v1);
    leg_apply<DAG, 2, TD, false, CH>(v2, U + 2 * 18, rr, ri);
    leg_load<P, DAG, 5, TD, O32>(in, nb[5], M, m, v2);
    leg_apply<DAG, 3, TD, false, CH>(v0, U + 3 * 18, rr, ri);
    leg_load<P, DAG, 6, TD, O32>(in, nb[6], M, m, v0);
    leg_apply<DAG, 4, TD, false, CH>(v1, U + 4 * 18, rr, ri);
    leg_load<P, DAG, 7, TD, O32>(in, nb[7], M, m, v1);
    leg_apply<DAG, 5, TD, false, CH>(v2, U + 5 * 18, rr, ri);
    leg_apply<DAG, 6, TD, false, CH>(v0, U + 6 * 18, rr, ri);
    leg_apply<DAG, 7, TD, false, CH>(v1, U + 7 * 18, rr, ri);
  } else {
    A v0[24], v1[24];
    leg_load<P, DAG, 0, TD, O32>(in, nb[0], M, m, v0);
    leg_load<P, DAG, 1, TD, O32>(in, nb[1], M, m, v1);
    leg_apply<DAG, 0, TD, true, CH>(v0, U + 0 * 18, rr, ri);
    leg_load<P, DAG, 2, TD, O32>(in, nb[2], M, m, v0);
    leg_apply<DAG, 1, TD, false, CH>(v1, U + 1 * 18, rr, ri);
    leg_load<P, DAG, 3, TD, O32>(in, nb[3], M, m, v1);
    leg_apply<DAG, 2, TD, false, CH>(v0, U + 2 * 18, rr, ri);
    leg_load<P, DAG, 4, TD, O32>(in, nb[4], M, m, v0);
    leg_apply<DAG, 3, TD, false, CH>(v1, U + 3 * 18, rr, ri);
    leg_load<P, DAG, 5, TD, O32>(in, nb[5], M, m, v1);
    leg_apply<DAG, 4, TD, false, CH>(v0, U + 4 * 18, rr, ri);
    leg_load<P, DAG, 6, TD, O32>(in, nb[6], M, m, v0);
    leg_apply<DAG, 5, TD, false, CH>(v1, U + 5 * 18, rr, ri);
    leg_load<P, DAG, 7, TD, O32>(in, nb[7], M, m, v1);
    leg_apply<DAG, 6, TD, false, CH>(v0, U + 6 * 18, rr, ri);
    leg_apply<DAG, 7, TD, false, CH>(v1, U + 7 * 18, rr, ri);
  }
}

// dhop_site on a domain part whose ghosts hold projected halves (load_nb_gp).
template <int P, bool DAG, int PF>
__device__ __forceinline__ void dhop_site_gp(const void *__restrict__ in, const uint32_t *nb, uint32_t M, uint32_t m,
                                             uint32_t ghost0, const typename Traits<P>::acc *U,
                                             typename Traits<P>::acc *rr, typename Traits<P>::acc *ri)
{
  typedef typename Traits<P>::acc A;
  constexpr int CH = MUL_CHAIN;
  if (PF == 0) {
    A v[24];
#define GBX_LEG(D, FIRST)                                                                  \
    {                                                                                      \
      const bool g = load_nb_gp<P>(in, nb[D], M, m, ghost0, v);                            \
      leg_compute_gp<LegProj<DAG, D>::value, FIRST, CH>(v, g, U + D * 18, rr, ri);         \
    }
    GBX_LEG(0, true)
    GBX_LEG(1, false)
    GBX_LEG(2, false)
    GBX_LEG(3, false)
    GBX_LEG(4, false)
    GBX_LEG(5, false)
    GBX_LEG(6, false)
    GBX_LEG(7, false)
#undef GBX_LEG
  } else if (PF == 2) {
    A v0[24], v1[24], v2[24];
    bool g0 = load_nb_gp<P>(in, nb[0], M, m, ghost0, v0);
    bool g1 = load_nb_gp<P>(in, nb[1], M, m, ghost0, v1);
    bool g2 = load_nb_gp<P>(in, nb[2], M, m, ghost0, v2);
    leg_compute_gp<LegProj<DAG, 0>::value, true, CH>(v0, g0, U + 0 * 18, rr, ri);
    g0 = load_nb_gp<P>(in, nb[3], M, m, ghost0, v0);
    leg_compute_gp<LegProj<DAG, 1>::value, false, CH>(v1, g1, U + 1 * 18, rr, ri);
    g1 = load_nb_gp<P>(in, nb[4], M, m, ghost0, v1);
    leg_compute_gp<LegProj<DAG, 2>::value, false, CH>(v2, g2, U + 2 * 18, rr, ri);
    g2 = load_nb_gp<P>(in, nb[5], M, m, ghost0, v2);
    leg_compute_gp<LegProj<DAG, 3>::value, false, CH>(v0, g0, U + 3 * 18, rr, ri);
    g0 = load_nb_gp<P>(in, nb[6], M, m, ghost0, v0);
    leg_compute_gp<LegProj<DAG, 4>::value, false, CH>(v1, g1, U + 4 * 18, rr, ri);
    g1 = load_nb_gp<P>(in, nb[7], M, m, ghost0, v1);
    leg_compute_gp<LegProj<DAG, 5>::value, false, CH>(v2, g2, U + 5 * 18, rr, ri);
    leg_compute_gp<LegProj<DAG, 6>::value, false, CH>(v0, g0, U + 6 * 18, rr, ri);
    leg_compute_gp<LegProj<DAG, 7>::value, false, CH>(v1, g1, U + 7 * 18, rr, ri);
  } else {
    A v0[24], v1[24];
    bool g0 = load_nb_gp<P>(in, nb[0], M, m, ghost0, v0);
    bool g1 = load_nb_gp<P>(in, nb[1], M, m, ghost0, v1);
    leg_compute_gp<LegProj<DAG, 0>::value, true, CH>(v0, g0, U + 0 * 18, rr, ri);
    g0 = load_nb_gp<P>(in, nb[2], M, m, ghost0, v0);
    leg_compute_gp<LegProj<DAG, 1>::value, false, CH>(v1, g1, U + 1 * 18, rr, ri);
    g1 = load_nb_gp<P>(in, nb[3], M, m, ghost0, v1);
    leg_compute_gp<LegProj<DAG, 2>::value, false, CH>(v0, g0, U + 2 * 18, rr, ri);
    g0 = load_nb_gp<P>(in, nb[4], M, m, ghost0, v0);
    leg_compute_gp<LegProj<DAG, 3>::value, false, CH>(v1, g1, U + 3 * 18, rr, ri);
    g1 = load_nb_gp<P>(in, nb[5], M, m, ghost0, v1);
    leg_compute_gp<LegProj<DAG, 4>::value, false, CH>(v0, g0, U + 4 * 18, rr, ri);
    g0 = load_nb_gp<P>(in, nb[6], M, m, ghost0, v0);
    leg_compute_gp<LegProj<DAG, 5>::value, false, CH>(v1, g1, U + 5 * 18, rr, ri);
    g1 = load_nb_gp<P>(in, nb[7], M, m, ghost0, v1);
    leg_compute_gp<LegProj<DAG, 6>::value, false, CH>(v0, g0, U + 6 * 18, rr, ri);
    leg_compute_gp<LegProj<DAG, 7>::value, false, CH>(v1, g1, U + 7 * 18, rr, ri);
  }
}

// Write the 4-spinor result (optionally out = alpha*center + beta*result,
// which then replaces the result in rr, ri).
template <int P, bool AXPBY>
__device__ __forceinline__ void store_site(void *__restrict__ out, const void *__restrict__ center, uint32_t q, uint32_t M,
                                           uint32_t m, typename Traits<P>::acc *rr, typename Traits<P>::acc *ri,
                                           typename Traits<P>::acc alpha, typename Traits<P>::acc beta, bool nt)
{
  typedef typename Traits<P>::acc A;
  constexpr int NCH = Traits<P>::NCH, R = Traits<P>::R;
  const uint64_t base = (uint64_t)q * NCH * M + m;
#pragma unroll
  for (int k = 0; k < NCH; k++) {
    A v[R];
#pragma unroll
    for (int j = 0; j < R; j++) {
      const int r = k * R + j;
      v[j] = (r & 1) ? ri[r >> 1] : rr[r >> 1];
    }
    if (AXPBY) {
      A c[R];
      load_chunk<P, A>(center, base + (uint64_t)k * M, c);
#pragma unroll
      for (int j = 0; j < R; j++) {
        const int r = k * R + j;
        v[j] = alpha * c[j] + beta * v[j];
        if (r & 1) ri[r >> 1] = v[j];
        else rr[r >> 1] = v[j];
      }
    }
    store_chunk<P, A>(out, base + (uint64_t)k * M, v, nt);
  }
}

}  // namespace dev
