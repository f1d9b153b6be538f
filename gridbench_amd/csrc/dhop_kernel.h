// The VALU hopping-term kernel template and its launch arguments, shared by
// the translation units that instantiate its forms: dhop.hip (plain, fused
// axpby, reference rounding, projected ghosts) and dhop_fused.hip (the solvers'
// fused operators).
#pragma once

#include "dhop_dev.h"
#include "gbx_internal.h"

namespace dhopk {

// What a workgroup does with its sites' results.
enum {
  EPI_STORE = 0,  // out = Dhop in
  EPI_AXPBY = 1,  // out = alpha c + beta Dhop in
  EPI_S5 = 2,     // out = Mooee c + beta Dhop in  (the adjoint of Mooee for DAG)
  EPI_S5INV = 3,  // out = Mooee^-1 Dhop in  (the adjoint for DAG)
  EPI_S5X = 4     // EPI_S5 in workgroups that hold whole columns of slices
};

// What it sums.
enum {
  RED_NONE = 0,
  RED_OUT = 1,   // |out|^2
  RED_RESID = 2  // r -= *a out in place of storing out, |r|^2
};

template <typename A> struct Epi {
  A alpha, beta;
  A d, mass;             // domain-wall terms: d = 5 - M5
  uint32_t Ls;
  const uint32_t *skip;  // nothing runs if *skip <= skip_at
  uint32_t skip_at;
  double *partial;       // the sum of every workgroup
  void *r;               // RED_RESID: a field of the arithmetic type
  const double *a;
};

// The residual's reals of chunks k0 .. k0+G-1 of a point (RED_RESID).
template <int P, int RED, int G>
__device__ __forceinline__ void load_resid(uint32_t q, uint32_t M, uint32_t m, int k0,
                                           const Epi<typename dev::Traits<P>::acc> &e, typename dev::Traits<P>::acc *x)
{
  typedef typename dev::Traits<P>::acc A;
  if constexpr (RED == RED_RESID) {
    constexpr int PR = P == GBX_F64 ? GBX_F64 : GBX_F32, RR = dev::Traits<PR>::R, RC = dev::Traits<PR>::NCH;
    constexpr int N = dev::Traits<P>::R / RR;
#pragma unroll
    for (int i = 0; i < G * N; i++) dev::load_chunk<PR, A>(e.r, ((uint64_t)q * RC + k0 * N + i) * M + m, x + i * RR);
  }
}

// The end of an epilogue for chunk k of a point: store it, or update the
// residual's reals x by it.
template <int P, int RED>
__device__ __forceinline__ void finish_chunk(void *__restrict__ out, uint32_t q, uint32_t M, uint32_t m, int k,
                                             const Epi<typename dev::Traits<P>::acc> &e, typename dev::Traits<P>::acc a,
                                             const typename dev::Traits<P>::acc *v, typename dev::Traits<P>::acc *x, bool nt,
                                             double &norm)
{
  typedef typename dev::Traits<P>::acc A;
  constexpr int NCH = dev::Traits<P>::NCH, R = dev::Traits<P>::R;
  if constexpr (RED == RED_RESID) {
    constexpr int PR = P == GBX_F64 ? GBX_F64 : GBX_F32, RR = dev::Traits<PR>::R, RC = dev::Traits<PR>::NCH, N = R / RR;
#pragma unroll
    for (int j = 0; j < R; j++) {
      x[j] -= a * v[j];
      norm += (double)x[j] * (double)x[j];
    }
#pragma unroll
    for (int i = 0; i < N; i++)
      dev::store_chunk<PR, A>(e.r, ((uint64_t)q * RC + k * N + i) * M + m, x + i * RR, false);
  } else {
    if constexpr (RED == RED_OUT) {
#pragma unroll
      for (int j = 0; j < R; j++) norm += (double)v[j] * (double)v[j];
    }
    dev::store_chunk<P, A>(out, ((uint64_t)q * NCH + k) * M + m, v, nt);
  }
}

// out = Mooee c + beta r for one (site, minor) point: the neighbour slice each
// chirality hops from (up in s for P-, down for P+, exchanged for DAG) is read
// from memory next to the point's own, mostly the same cache lines.
template <int P, bool DAG, int RED>
__device__ __forceinline__ void store_s5(void *__restrict__ out, const void *__restrict__ c, uint32_t q, uint32_t M, uint32_t m,
                                         const Epi<typename dev::Traits<P>::acc> &e, typename dev::Traits<P>::acc *rr,
                                         typename dev::Traits<P>::acc *ri, bool nt, double &norm)
{
  typedef typename dev::Traits<P>::acc A;
  constexpr int NCH = dev::Traits<P>::NCH, R = dev::Traits<P>::R;
  __builtin_amdgcn_sched_barrier(0);  // c's chunks are not held across the legs
  const uint64_t base = (uint64_t)q * NCH * M;
  const uint32_t s = m % e.Ls;
  const uint32_t mdn = s == 0 ? m + e.Ls - 1 : m - 1, mup = s == e.Ls - 1 ? m - (e.Ls - 1) : m + 1;
  const A cdn = s == 0 ? e.mass : (A)-1, cup = s == e.Ls - 1 ? e.mass : (A)-1;
  const A a = RED == RED_RESID ? (A)*e.a : (A)0;
#pragma unroll
  for (int k = 0; k < NCH; k++) {
    if (R == 8) __builtin_amdgcn_sched_barrier(0);  // one 16-bit chunk at a time: 3 or 4 loads of 8 reals
    A own[R], dn[R], up[R], v[R], x[R];
    const bool has_dn = DAG ? (k + 1) * R > 12 : k * R < 12, has_up = DAG ? k * R < 12 : (k + 1) * R > 12;
    dev::load_chunk<P, A>(c, base + (uint64_t)k * M + m, own);
    if (has_dn) dev::load_chunk<P, A>(c, base + (uint64_t)k * M + mdn, dn);
    if (has_up) dev::load_chunk<P, A>(c, base + (uint64_t)k * M + mup, up);
    load_resid<P, RED, 1>(q, M, m, k, e, x);
#pragma unroll
    for (int j = 0; j < R; j++) {
      const int r = k * R + j;
      const bool down = (r < 12) != DAG;
      const A acc = e.d * own[j] + (down ? cdn : cup) * (down ? dn[j] : up[j]);
      v[j] = acc + e.beta * ((r & 1) ? ri[r >> 1] : rr[r >> 1]);
    }
    finish_chunk<P, RED>(out, q, M, m, k, e, a, v, x, nt, norm);
  }
}

// store_s5 for a workgroup that holds whole (site, right-hand side) columns of
// Ls slices, one point per thread: each thread reads its own slice of c only
// and takes the neighbour slices from LDS, a chirality at a time (16-bit
// fields all three chunks at once).  Half the loads of store_s5 and fewer
// registers (FP32 72 instead of 81, 73 instead of 96 with the norm: 7 or 6
// wavefronts a SIMD instead of 5).  What bounds the kernel is still the legs'
// gathers: 24^4 x Ls16 FP64 869 -> 863 us, the domain-wall solve at 16^4 x
// Ls12, FP32 inner, 16.40 -> 16.28 ms.  Every thread calls it; `w` is the
// point's index in the workgroup, s its slice, `active` whether it has one.
template <int P, bool DAG, int RED>
__device__ __forceinline__ void store_s5x(void *__restrict__ out, const void *__restrict__ c, uint32_t q, uint32_t M, uint32_t m,
                                          const Epi<typename dev::Traits<P>::acc> &e, uint32_t w, uint32_t s, bool active,
                                          unsigned char *smem, typename dev::Traits<P>::acc *rr,
                                          typename dev::Traits<P>::acc *ri, bool nt, double &norm)
{
  typedef typename dev::Traits<P>::acc A;
  typedef typename dev::Traits<P>::vec V;
  constexpr int NCH = dev::Traits<P>::NCH, R = dev::Traits<P>::R, G = R == 8 ? NCH : NCH / 2;
  V *sx = (V *)smem;  // [G][threads]
  const uint64_t base = (uint64_t)q * NCH * M + m;
  const uint32_t th = blockDim.x;
  const uint32_t wdn = s == 0 ? w + e.Ls - 1 : w - 1, wup = s == e.Ls - 1 ? w - (e.Ls - 1) : w + 1;
  const A cdn = s == 0 ? e.mass : (A)-1, cup = s == e.Ls - 1 ? e.mass : (A)-1;
  const A a = RED == RED_RESID ? (A)*e.a : (A)0;
#pragma unroll
  for (int k0 = 0; k0 < NCH; k0 += G) {
    V own[G];
    A x[G * R];
    __builtin_amdgcn_sched_barrier(0);  // c's chunks are not held across the legs
    if (active) {
#pragma unroll
      for (int k = 0; k < G; k++) own[k] = ((const V *)c)[base + (uint64_t)(k0 + k) * M];
      load_resid<P, RED, G>(q, M, m, k0, e, x);
    }
    __syncthreads();  // the links, or the other chirality, are no longer read
    if (active) {
#pragma unroll
      for (int k = 0; k < G; k++) sx[k * th + w] = own[k];
    }
    __syncthreads();
    if (active) {
#pragma unroll
      for (int k = 0; k < G; k++) {
        __builtin_amdgcn_sched_barrier(0);  // one chunk's reals at a time
        const int r0 = (k0 + k) * R;
        const bool has_dn = DAG ? r0 + R > 12 : r0 < 12, has_up = DAG ? r0 < 12 : r0 + R > 12;
        V dn, up;
        A v[R];
        if (has_dn) dn = sx[k * th + wdn];
        if (has_up) up = sx[k * th + wup];
#pragma unroll
        for (int j = 0; j < R; j++) {
          const int r = r0 + j;
          const bool down = (r < 12) != DAG;
          const A acc = e.d * (A)own[k][j] + (down ? cdn : cup) * (A)(down ? dn[j] : up[j]);
          v[j] = acc + e.beta * ((r & 1) ? ri[r >> 1] : rr[r >> 1]);
        }
        finish_chunk<P, RED>(out, q, M, m, k0 + k, e, a, v, x + k * R, nt, norm);
      }
    }
  }
}

// r = Mooee^-1 r (closed form, see k_dwf_s5_inv in dwf.hip) for the points of a
// workgroup that holds whole (site, right-hand side) columns of Ls slices, one
// point per thread: the reals of one chirality at a time through LDS, each
// column in the order its shift walks it.  Every thread calls it; `w` is the
// point's index in the workgroup, s its slice, `active` whether it has one.
template <bool DAG, typename A>
__device__ __forceinline__ void s5_inverse(const Epi<A> &e, uint32_t w, uint32_t s, bool active, unsigned char *smem, A *rr,
                                           A *ri)
{
  constexpr int SV = 16 / sizeof(A), N = 12 / SV;  // reals of an LDS entry, entries of a chirality
  typedef A AV __attribute__((ext_vector_type(SV)));
  AV *sx = (AV *)smem;  // [N][threads]
  const uint32_t nt = blockDim.x, Ls = e.Ls;
  const A dinv = (A)1 / e.d;
  A dls = (A)1;
  for (uint32_t k = 0; k < Ls; k++) dls *= dinv;
  const A gnorm = (A)1 / ((A)1 + e.mass * dls);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const bool down = (h == 0) != DAG;
    const uint32_t pos = down ? s : Ls - 1 - s, col = w - s;
    __syncthreads();  // the links, or the other chirality, are no longer read
    if (active) {
#pragma unroll
      for (int j = 0; j < N; j++) {
        AV x;
#pragma unroll
        for (int i = 0; i < SV; i++) {
          const int r = h * 12 + j * SV + i;
          x[i] = (r & 1) ? ri[r >> 1] : rr[r >> 1];
        }
        sx[j * nt + col + pos] = x;
      }
    }
    __syncthreads();
    if (active) {
      A acc[12];
#pragma unroll
      for (int i = 0; i < 12; i++) acc[i] = (A)0;
      A wk = dinv;
      for (uint32_t k = 0; k < Ls; k++) {
        const bool wrap = k > pos;
        const A c = wrap ? -e.mass * wk : wk;
        const AV *x = sx + col + pos - k + (wrap ? Ls : 0);
#pragma unroll
        for (int j = 0; j < N; j++) {
          const AV v = x[j * nt];
#pragma unroll
          for (int i = 0; i < SV; i++) acc[j * SV + i] += c * v[i];
        }
        wk *= dinv;
      }
#pragma unroll
      for (int i = 0; i < 12; i++) {
        const int r = h * 12 + i;
        if (r & 1) ri[r >> 1] = acc[i] * gnorm;
        else rr[r >> 1] = acc[i] * gnorm;
      }
    }
  }
}

// A point's site and minor index once more: not kept in registers across the
// legs.
__device__ __forceinline__ void again(uint32_t &w, uint32_t mcc, uint32_t &sl, uint32_t &m)
{
  asm volatile("" : "+v"(w));
  sl = w / mcc;
  m = w - sl * mcc;
}

// alpha c + beta r of one point and its sum, a chunk at a time: with
// all 24 results and their squares in registers together the 16-bit forms need
// more than the plain kernel's 80 and lose a wavefront of six.  CG at 16^3x24
// x Ls8, FP16 inner: 13.6 -> 13.1 ms.
template <int P, int RED>
__device__ __forceinline__ void store_axpby_norm(void *__restrict__ out, const void *__restrict__ c, uint32_t q, uint32_t M,
                                                 uint32_t m, const Epi<typename dev::Traits<P>::acc> &e,
                                                 typename dev::Traits<P>::acc *rr, typename dev::Traits<P>::acc *ri, bool nt,
                                                 double &norm)
{
  typedef typename dev::Traits<P>::acc A;
  typedef typename dev::Traits<P>::vec V;
  constexpr int NCH = dev::Traits<P>::NCH, R = dev::Traits<P>::R, G = NCH < 6 ? NCH : NCH / 2;
  const uint64_t base = (uint64_t)q * NCH * M + m;
  const A a = RED == RED_RESID ? (A)*e.a : (A)0;
#pragma unroll
  for (int k0 = 0; k0 < NCH; k0 += G) {
    V own[G];
    A x[G * R];
    __builtin_amdgcn_sched_barrier(0);  // c's chunks are not held across the legs
#pragma unroll
    for (int k = 0; k < G; k++) own[k] = ((const V *)c)[base + (uint64_t)(k0 + k) * M];
    load_resid<P, RED, G>(q, M, m, k0, e, x);
#pragma unroll
    for (int k = 0; k < G; k++) {
      __builtin_amdgcn_sched_barrier(0);
      A v[R];
#pragma unroll
      for (int j = 0; j < R; j++) {
        const int r = (k0 + k) * R + j;
        v[j] = e.alpha * (A)own[k][j] + e.beta * ((r & 1) ? ri[r >> 1] : rr[r >> 1]);
      }
      finish_chunk<P, RED>(out, q, M, m, k0 + k, e, a, v, x + k * R, nt, norm);
    }
  }
}

// Sum over the workgroup in a fixed order (at most 16 wavefronts).
__device__ __forceinline__ double block_sum(double a)
{
  __shared__ double sh[16];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = a;
  __syncthreads();
  double t = 0.0;
  for (uint32_t i = 0; i < blockDim.x >> 6; i++) t += sh[i];
  return t;
}

// Logical workgroup L covers sites q0 .. q0+spw-1 (site block L % nwg_sites)
// and minor indices m0 .. m0+mc-1 (minor chunk L / nwg_sites): with mc < M
// the lattice is swept once per minor chunk, so the 8-neighbour working set
// is that of an mc-wide field (the links are re-read once per chunk).
// GP: a domain part whose ghosts hold spin-projected halves from ghost0 on
// (dhop_site_gp).  TD: fields in the GBX_BASIS_TDIAG spin basis.  RED: also a
// sum over the workgroup's values (RED_OUT: before their rounding to the
// storage precision) into e.partial[L], in FP64 and a fixed order.  O32: 32-bit
// gather offsets (dev::load_at).
template <int P, bool DAG, bool C12, int EPI, int PF, bool EXACT, bool GP, bool TD, int RED, bool O32>
__global__ void __launch_bounds__(PF ? 256 : 1024)
    k_dhop(const void *__restrict__ gauge, const uint32_t *__restrict__ nbr, const void *__restrict__ in,
           void *__restrict__ out, const void *__restrict__ center, uint32_t nslot, uint32_t M, uint32_t spw, uint32_t mc,
           uint32_t nwg_sites, uint32_t cblk, uint32_t nchunk, uint32_t nwg, uint32_t per_xcd, int xcd, int nt,
           Epi<typename dev::Traits<P>::acc> e, uint32_t ghost0)
{
  typedef typename dev::Traits<P>::acc A;
  extern __shared__ __align__(16) unsigned char smem[];
  A *sU = (A *)smem;
  uint32_t *sN = (uint32_t *)(sU + (size_t)spw * 8 * 18);

  const uint32_t L = xcd ? (blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3) : blockIdx.x;
  if (L >= nwg) return;  // uniform over the workgroup, before any barrier
  if (e.skip && *e.skip <= e.skip_at) return;
  // cblk site groups are visited for every minor chunk before the next
  // cblk groups (chunk-inner order); cblk == nwg_sites sweeps the lattice
  // once per chunk (chunk-outer order).
  const uint32_t per = cblk * nchunk, grp = L / per, r = L - grp * per;
  const uint32_t chunk = r / cblk, b = grp * cblk + (r - chunk * cblk);
  if (b >= nwg_sites) {
    if constexpr (RED) {
      if (threadIdx.x == 0) e.partial[L] = 0.0;
    }
    return;
  }
  const uint32_t q0 = b * spw, m0 = chunk * mc;
  const uint32_t nsl = min(spw, nslot - q0), mcc = min(mc, M - m0);
  dev::stage_links<P, C12>(gauge, nbr, q0, nsl, sU, sN, O32 ? dev::Traits<P>::NCH * M * 16 : 1);

  const uint32_t items = nsl * mcc;
  if constexpr (EPI == EPI_S5INV || EPI == EPI_S5X) {  // one point per thread, whole columns
    uint32_t w = threadIdx.x, sl = w / mcc, m = w - sl * mcc;
    const bool active = w < items;
    A rr[12], ri[12];
    if (active) {
      dev::dhop_site<P, DAG, PF, EXACT, TD, O32>(in, sN + sl * 8, M, m, sU + sl * 8 * 18, rr, ri);
      dev::pin_acc(rr, ri);
    }
    again(w, mcc, sl, m);
    if constexpr (EPI == EPI_S5X) {
      double norm = 0.0;
      store_s5x<P, DAG, RED>(out, center, q0 + sl, M, m, e, w, m % e.Ls, active, smem, rr, ri, nt != 0, norm);
      if constexpr (RED) {
        norm = block_sum(norm);
        if (threadIdx.x == 0) e.partial[L] = norm;
      }
      return;
    }
    s5_inverse<DAG>(e, w, m % e.Ls, active, smem, rr, ri);
    if (active) dev::store_site<P, false>(out, nullptr, q0 + sl, M, m, rr, ri, (A)0, (A)1, nt != 0);
    return;
  }
  double norm = 0.0;
  for (uint32_t w = threadIdx.x; w < items; w += blockDim.x) {
    uint32_t sl = w / mcc, m = m0 + (w - sl * mcc);
    A rr[12], ri[12];
    if constexpr (GP) dev::dhop_site_gp<P, DAG, PF>(in, sN + sl * 8, M, m, ghost0, sU + sl * 8 * 18, rr, ri);
    else dev::dhop_site<P, DAG, PF, EXACT, TD, O32>(in, sN + sl * 8, M, m, sU + sl * 8 * 18, rr, ri);
    if constexpr (EPI == EPI_AXPBY && RED) {
      uint32_t w2 = w;
      dev::pin_acc(rr, ri);
      again(w2, mcc, sl, m);
      m += m0;
    }
    if constexpr (EPI == EPI_S5) store_s5<P, DAG, RED>(out, center, q0 + sl, M, m, e, rr, ri, nt != 0, norm);
    else if constexpr (RED) store_axpby_norm<P, RED>(out, center, q0 + sl, M, m, e, rr, ri, nt != 0, norm);
    else dev::store_site<P, EPI == EPI_AXPBY>(out, center, q0 + sl, M, m, rr, ri, e.alpha, e.beta, nt != 0);
  }
  if constexpr (RED) {
    norm = block_sum(norm);
    if (threadIdx.x == 0) e.partial[L] = norm;
  }
}

struct LaunchArgs {
  dim3 grid, block;
  size_t lds;
  hipStream_t st;
  const void *gauge;
  const uint32_t *nbr;
  const void *in;
  void *out;
  const void *center;
  uint32_t nslot, M, spw, mc, nwg_sites, cblk, nchunk, nwg, per_xcd;
  int xcd, nt;
  double alpha, beta;
  uint32_t ghost0;
  double d = 0, mass = 0;
  uint32_t Ls = 1;
  const uint32_t *skip = nullptr;
  uint32_t skip_at = 0;
  double *partial = nullptr;
  void *r = nullptr;
  const double *a = nullptr;
  uint64_t in_bytes = 0;
};

template <int P, bool DAG, bool C12, int EPI, int PF, bool EXACT = false, bool GP = false, bool TD = false, int RED = RED_NONE>
void launch_t(const LaunchArgs &a)
{
  typedef typename dev::Traits<P>::acc A;
  const Epi<A> e{(A)a.alpha, (A)a.beta, (A)a.d, (A)a.mass, a.Ls, a.skip, a.skip_at, a.partial, a.r, a.a};
  auto *k = &k_dhop<P, DAG, C12, EPI, PF, EXACT, GP, TD, RED, false>;
  if constexpr (P != GBX_F64 && (EPI >= EPI_S5 || RED != RED_NONE)) {
    if (a.in_bytes <= (1ull << 32)) k = &k_dhop<P, DAG, C12, EPI, PF, EXACT, GP, TD, RED, true>;
  }
  hipLaunchKernelGGL(k, a.grid, a.block, a.lds, a.st, a.gauge, a.nbr, a.in, a.out, a.center, a.nslot, a.M, a.spw, a.mc,
                     a.nwg_sites, a.cblk, a.nchunk, a.nwg, a.per_xcd, a.xcd, a.nt, e, a.ghost0);
}

// The fused forms (dhop_fused.hip): the fifth-dimension epilogues and the
// forms that also sum (RED_OUT without, RED_RESID with dag).
void launch_fused(int prec, int epi, bool dag, bool c12, bool td, int red, int pf, const LaunchArgs &a);

}  // namespace dhopk
