// Defect-correction conjugate gradient for  M^dagger M x = b,
// M = 1 - kappa Dhop  (M^dagger = 1 - kappa Dhop^dagger), and the even-odd
// (Schur complement) solve of M x = b on a red-black pair: with
// Mpc = 1 - kappa^2 DhopEO DhopOE on the even sites the outer loop works on
// r = b'_e - Mpc x_e and the inner CG on Mpc^dag Mpc (CGNR).
//
// Outer loop, FP64 on the GPU:
//   r = b - M^dag M x  (FP64 hopping kernels; the "true" residual)
//   stop when |r| / |b| <= tol
//   r_in = s * r with s = sqrt(N) / |r|  (unit-RMS entries: safe for FP16)
//   e = inner_solve(M_lo^dag M_lo e = r_in) to |r_in - ...| <= inner_tol |r_in|
//   x += e / s          (reliable update of x in FP64)
// Inner CG: vectors e, r in FP32; p and t = M p in the low storage precision of
// the inner gauge field (FP32, FP16 or BF16), which is what the low-precision
// hopping kernel reads and writes; every arithmetic operation in FP32; dots
// and norms in FP64 with deterministic reductions.  With A = M^dag M one
// iteration is
//   t = M p, and <p, A p> = |t|^2 summed by the kernel that writes t
//   k_cg_alpha:  a = |r_old|^2 / |t|^2
//   r -= a M^dag t and |r|^2 in the epilogue of the kernel that forms M^dag t,
//     which is never stored
//   k_cg_ep: p = r + b p (b = |r|^2 / |r_old|^2), and every other iteration
//     e += a' p' + a p for the last two
// The scalars stay on the device, so no kernel waits for the host.  The host
// enqueues a few iterations ahead and learns of convergence from a word the
// device writes to its memory; what was enqueued beyond it does nothing.
// An iteration at 16^3x24 x Ls8, FP16 inner, takes 111 us with no gaps: 33 us
// for M p, 39 us for M^dag t with the update of r, 5 us for k_cg_alpha, and 23
// or 46 us for k_cg_ep (6 TB/s).  It took 307 us with the two sums read back by
// the host and the updates in passes of their own, and 163 us with the scalars
// on the device but M^dag t stored and read again (30 us) and e updated each
// time (42 us): 13.6 -> 12.0 ms a solve (9.7 since the hops stage their links
// in one round trip); domain-wall solve 16^4 x Ls12, FP32 inner: 16.3 -> 15.2
// ms (13.5).  The partial sums are summed where they are needed
// up to kPlain of them, which costs a reader 2 us; a pass of its own takes 5.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <mutex>
#include <vector>

#include "dhop_dev.h"
#include "gbx_internal.h"

namespace {

// Workgroups and threads of a pass over a field; partial sums beyond kPlain
// are folded into kFold first.
constexpr int kRB = 1024, kRT = 256, kAT = 1024, kPlain = 8192, kFold = 256;

template <int P> struct Pt {
  typedef typename dev::Traits<P>::acc A;
  static constexpr int R = dev::Traits<P>::R, NCH = dev::Traits<P>::NCH;
};

template <int P, typename A>
__device__ __forceinline__ void load_pt(const void *b, uint64_t q, uint32_t M, uint32_t m, A *v)
{
#pragma unroll
  for (int k = 0; k < Pt<P>::NCH; k++) dev::load_chunk<P, A>(b, (q * Pt<P>::NCH + k) * M + m, v + k * Pt<P>::R);
}

template <int P, typename A>
__device__ __forceinline__ void store_pt(void *b, uint64_t q, uint32_t M, uint32_t m, const A *v)
{
#pragma unroll
  for (int k = 0; k < Pt<P>::NCH; k++) dev::store_chunk<P, A>(b, (q * Pt<P>::NCH + k) * M + m, v + k * Pt<P>::R, false);
}

// Sum over the workgroup of T threads in a fixed order; every thread gets it.
template <int T = kRT>
__device__ __forceinline__ double bsum(double a)
{
  __shared__ double sh[T / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, 64);
  __syncthreads();  // an earlier sum has been read
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = a;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int i = 0; i < T / 64; i++) t += sh[i];
  return t;
}

// Sum of n partial sums, by every workgroup on its own.
template <int T = kRT>
__device__ __forceinline__ double sum_partials(const double *__restrict__ part, int n)
{
  double a = 0.0;
#pragma unroll 8
  for (int i = threadIdx.x; i < n; i += T) a += part[i];
  return bsum<T>(a);
}

// The inner solve's scalars.  rr[i & 1] is |r|^2 at iteration i (two, so that
// the workgroups of k_cg_ep can read the old one while the new one is
// written), alpha[i & 1] its step; iteration i and later do nothing once
// done_at <= i, nor the rest of an iteration that breaks off once hop_at <= i.
struct CgScal {
  double rr[2], alpha[2], stop;
  uint32_t done_at, hop_at, iters, broke;
};

// What the host learns after every iteration that ran, in one word of its own
// memory: the iterations behind it, whether the solve ended, and whether it
// ended without an update (<p, A p> not positive: the accuracy floor).
__device__ __forceinline__ void tell_host(uint64_t *word, uint32_t seq, bool done, bool broke)
{
  const uint64_t v = (uint64_t)seq | (done ? 1ull << 32 : 0) | (broke ? 1ull << 33 : 0);
  __hip_atomic_store(word, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// r = scale * src, p = r, partial |r|^2.
template <int PE, int PP>
__global__ void __launch_bounds__(kRT) k_cg_start(double scale, const void *__restrict__ src, void *__restrict__ r,
                                                  void *__restrict__ p, uint64_t npts, uint32_t M, double *__restrict__ partial)
{
  typedef typename Pt<PE>::A A;
  double acc = 0.0;
  for (uint64_t t = blockIdx.x * (uint64_t)kRT + threadIdx.x; t < npts; t += (uint64_t)gridDim.x * kRT) {
    const uint64_t q = t / M;
    const uint32_t m = (uint32_t)(t % M);
    double sv[24];
    A rv[24];
    load_pt<GBX_F64, double>(src, q, M, m, sv);
#pragma unroll
    for (int j = 0; j < 24; j++) {
      rv[j] = (A)(sv[j] * scale);
      acc += (double)rv[j] * (double)rv[j];
    }
    store_pt<PE, A>(r, q, M, m, rv);
    store_pt<PP, A>(p, q, M, m, rv);
  }
  acc = bsum(acc);
  if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

__global__ void __launch_bounds__(kRT) k_cg_begin(CgScal *__restrict__ s, const double *__restrict__ partial, int n, double rel_tol)
{
  const double rr = sum_partials(partial, n);
  if (threadIdx.x == 0) {
    s->rr[0] = rr;
    s->stop = rel_tol * rel_tol * rr;
    s->alpha[0] = s->alpha[1] = 0.0;
    s->done_at = s->hop_at = 0xffffffffu;
    s->iters = s->broke = 0;
  }
}

// n partial sums into gridDim.x of them.
__global__ void __launch_bounds__(kRT) k_cg_fold(const CgScal *__restrict__ s, uint32_t it, const double *__restrict__ in, int n,
                                                 double *__restrict__ out)
{
  if (s->done_at <= it) return;
  double a = 0.0;
  for (int i = blockIdx.x * kRT + threadIdx.x; i < n; i += gridDim.x * kRT) a += in[i];
  a = bsum(a);
  if (threadIdx.x == 0) out[blockIdx.x] = a;
}

// a = |r|^2 / |t|^2 from the partial sums of |t|^2, by one workgroup.  |t|^2 not
// positive (the accuracy floor): iteration `it` ends without an update.
__global__ void __launch_bounds__(kAT) k_cg_alpha(CgScal *__restrict__ s, uint32_t it, const double *__restrict__ tt, int n)
{
  if (s->done_at <= it) return;
  const double pap = sum_partials<kAT>(tt, n);
  if (threadIdx.x == 0) {
    const bool ok = pap > 0.0;
    s->alpha[it & 1] = ok ? s->rr[it & 1] / pap : 0.0;
    if (!ok) {
      s->broke = 1u;
      s->hop_at = it;
    }
  }
}

// p' = r + b p and the iteration's outcome; e is brought up to date every other
// iteration and at the end: PAIR: e += a' q + a p with q, a' the last
// iteration's p and a, and p' goes over q.  Otherwise p' goes to another field,
// p and a are left to the next iteration, or if it is the last: e += a p and
// no p'.  first: e = ... instead of e += ...
template <int PE, int PP, bool PAIR>
__global__ void __launch_bounds__(kRT) k_cg_ep(CgScal *__restrict__ s, uint32_t it, const double *__restrict__ rpart, int nr,
                                               const void *__restrict__ r, const void *__restrict__ p, void *pn,
                                               void *__restrict__ e, uint64_t npts, uint32_t M, int first, int last,
                                               uint64_t *word)
{
  typedef typename Pt<PE>::A A;
  if (s->done_at <= it) return;
  const bool broke = s->broke != 0;
  double rr_new = 0.0, b = 0.0;
  bool done = true;
  if (!broke) {
    rr_new = sum_partials<kRT>(rpart, nr);
    b = rr_new / s->rr[it & 1];
    done = !(rr_new > s->stop);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (!broke) {
      s->rr[(it + 1) & 1] = rr_new;
      s->iters = it + 1;
    }
    if (done) s->done_at = s->hop_at = it + 1;
    tell_host(word, it + 1, done, broke);
  }
  const bool end = done || last;
  if (broke && !PAIR) return;
  const A a = broke ? (A)0 : (A)s->alpha[it & 1], a1 = PAIR ? (A)s->alpha[(it + 1) & 1] : (A)0;
  for (uint64_t t = blockIdx.x * (uint64_t)kRT + threadIdx.x; t < npts; t += (uint64_t)gridDim.x * kRT) {
    const uint64_t q = t / M;
    const uint32_t m = (uint32_t)(t % M);
    A pv[24], v[24];
    load_pt<PP, A>(p, q, M, m, pv);
    if (PAIR || end) {
      A ev[24];
      if (!first) load_pt<PE, A>(e, q, M, m, ev);
      if (PAIR) load_pt<PP, A>(pn, q, M, m, v);
#pragma unroll
      for (int j = 0; j < 24; j++) {
        ev[j] = first ? (A)0 : ev[j];
        if (PAIR) ev[j] += a1 * v[j];
        if (!broke) ev[j] += a * pv[j];
      }
      store_pt<PE, A>(e, q, M, m, ev);
    }
    if (!end) {
      load_pt<PE, A>(r, q, M, m, v);
#pragma unroll
      for (int j = 0; j < 24; j++) v[j] += (A)b * pv[j];
      store_pt<PP, A>(pn, q, M, m, v);
    }
  }
}

// z = a x + b y on FP64 fields, partial |z|^2.
__global__ void __launch_bounds__(kRT) k_axpby_norm(double a, const void *__restrict__ x, double b, const void *__restrict__ y,
                                                    void *__restrict__ z, uint64_t nchunk, double *__restrict__ partial)
{
  double acc = 0.0;
  for (uint64_t t = blockIdx.x * (uint64_t)kRT + threadIdx.x; t < nchunk; t += (uint64_t)gridDim.x * kRT) {
    double xv[2], yv[2];
    dev::load_chunk<GBX_F64, double>(x, t, xv);
    dev::load_chunk<GBX_F64, double>(y, t, yv);
#pragma unroll
    for (int j = 0; j < 2; j++) {
      xv[j] = a * xv[j] + b * yv[j];
      acc += xv[j] * xv[j];
    }
    dev::store_chunk<GBX_F64, double>(z, t, xv, false);
  }
  acc = bsum(acc);
  if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

// x (FP64) += a e (precision PS)
template <int PS>
__global__ void __launch_bounds__(kRT) k_axpy_into_f64(double a, const void *__restrict__ e, void *__restrict__ x, uint64_t npts,
                                                       uint32_t M)
{
  for (uint64_t t = blockIdx.x * (uint64_t)kRT + threadIdx.x; t < npts; t += (uint64_t)gridDim.x * kRT) {
    const uint64_t q = t / M;
    const uint32_t m = (uint32_t)(t % M);
    double ev[24], xv[24];
    load_pt<PS, double>(e, q, M, m, ev);
    load_pt<GBX_F64, double>(x, q, M, m, xv);
#pragma unroll
    for (int j = 0; j < 24; j++) xv[j] += a * ev[j];
    store_pt<GBX_F64, double>(x, q, M, m, xv);
  }
}

// Sum of partial sums, written to the host's memory.
__global__ void __launch_bounds__(kRT) k_final(const double *__restrict__ partial, int n, double *out)
{
  const double a = sum_partials(partial, n);
  if (threadIdx.x == 0) out[0] = a;
}

// Pinned host memory of a solve: the word the device reports iterations in, and
// a sum.  A solve takes one for itself and gives it back; up to kWords unused
// ones are kept for later solves.
struct HostWords {
  uint64_t word;
  double sum;
};

constexpr size_t kWords = 8;
std::mutex g_words_mu;
std::vector<HostWords *> g_words;

int take_words(HostWords **w)
{
  {
    std::lock_guard<std::mutex> lk(g_words_mu);
    if (!g_words.empty()) {
      *w = g_words.back();
      g_words.pop_back();
      return GBX_OK;
    }
  }
  GBX_HIP(hipHostMalloc(w, sizeof(HostWords), hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent));
  return GBX_OK;
}

void give_words(HostWords *w)
{
  {
    std::lock_guard<std::mutex> lk(g_words_mu);
    if (g_words.size() < kWords) {
      g_words.push_back(w);
      return;
    }
  }
  (void)hipHostFree(w);
}

// Device memory of one solve: its fields and scalars in one allocation (eight
// of them, freed one by one, cost 2.3 ms of an 18 ms solve).
struct Workspace {
  char *base = nullptr;
  size_t bytes = 0;
  hipStream_t st = nullptr;
  std::vector<gbx_spinor_s *> fields;
  std::vector<size_t> at;
  HostWords *words = nullptr;
  ~Workspace()
  {
    if (base) {
      (void)hipStreamSynchronize(st);
      (void)hipFree(base);
    }
    if (words) give_words(words);  // no kernel writes to them any more
  }
  size_t take(size_t n)
  {
    const size_t o = bytes;
    bytes += (n + 255) & ~(size_t)255;
    return o;
  }
  // A field of Ls slices and one right-hand side on g, in basis `basis`.
  void field(gbx_spinor_s &f, gbx_geom_s *g, int Ls, int prec, int basis)
  {
    f.geom = g;
    f.Ls = Ls;
    f.nrhs = 1;
    f.prec = prec;
    f.M = (uint32_t)Ls;
    f.bytes = (g->vol + g->nghost) * (size_t)Ls * 24 * (size_t)prec_bytes(prec);
    f.basis = basis;
    fields.push_back(&f);
    at.push_back(take(f.bytes));
  }
  int allocate(hipStream_t s)
  {
    st = s;
    if (hipMalloc(&base, bytes) != hipSuccess) {
      (void)hipGetLastError();
      base = nullptr;
      return gbx_fail(GBX_ENOMEM, "cg: cannot allocate %zu bytes of workspace", bytes);
    }
    for (size_t i = 0; i < fields.size(); i++) fields[i]->d = base + at[i];
    return GBX_OK;
  }
};

// The scalars and partial sums of a solve.
struct Scratch {
  size_t scal_at = 0, part_at = 0, tt_at = 0, fold_at = 0;
  CgScal *scal = nullptr;
  double *partial = nullptr, *tt = nullptr, *fold = nullptr;
  HostWords *host = nullptr;
  void plan(Workspace &w, uint32_t ntt)
  {
    scal_at = w.take(sizeof(CgScal));
    part_at = w.take(sizeof(double) * kRB);
    tt_at = w.take(sizeof(double) * ntt);
    fold_at = w.take(sizeof(double) * kFold);
  }
  int init(Workspace &w)
  {
    scal = (CgScal *)(w.base + scal_at);
    partial = (double *)(w.base + part_at);
    tt = (double *)(w.base + tt_at);
    fold = (double *)(w.base + fold_at);
    GBX_TRY(take_words(&w.words));
    host = w.words;
    return GBX_OK;
  }
  // The sum of n partial sums on the host (waits for the stream).
  int fetch(hipStream_t st, int n, double *v)
  {
    hipLaunchKernelGGL(k_final, dim3(1), dim3(kRT), 0, st, (const double *)partial, n, &host->sum);
    GBX_HIP(hipGetLastError());
    GBX_HIP(hipStreamSynchronize(st));
    *v = host->sum;
    return GBX_OK;
  }
};

// Workgroups of a pass over n elements (its partial sums).
int blocks_for(uint64_t n) { return (int)std::min<uint64_t>((n + kRT - 1) / kRT, kRB); }

// Launch configuration of the solver's hopping kernels: the tuned VALU
// configuration of this signature (the fused forms run on the VALU kernel)
// with cached output stores, since the solver reads its outputs back at once.
dhop_cfg solver_cfg(const gbx_gauge_s *u, const gbx_spinor_s *in)
{
  dhop_cfg c = dhop_fused_cfg(u, in);
  c.nt = 0;
  return c;
}

// The positive operator A the CG inverts, with its temporaries:
//   whole lattice:  A = M^dag M        (u = the lattice's gauge field, t)
//   red-black pair: A = Mpc^dag Mpc     (ue / uo = even / odd halves' fields,
//                   t on the even half, to on the odd half)
enum { OP_WILSON = 0, OP_DWF = 1 };

struct NormalOp {
  bool eo;
  const gbx_gauge_s *ue, *uo;
  double kappa;
  gbx_spinor_s *t, *to;
  int kind = OP_WILSON;       // red-black only: M = 1 - kappa Dhop, or the DWF operator
  gbx_dwf_params dwf{0, 0};
  dhop_cfg ce{}, co{};         // launch shapes of the hops on ue and uo
  void shapes()
  {
    ce = solver_cfg(ue, t);
    if (eo) co = solver_cfg(uo, t);
  }
};

// An application inside the inner CG: it does nothing once *skip <= skip_at, and
// its last kernel sums into `partial`: of M, |out|^2; of M^dag, |r|^2 after
// r -= *a out in place of writing out.
struct Step {
  const uint32_t *skip = nullptr;
  uint32_t skip_at = 0;
  double *partial = nullptr;
  gbx_spinor_s *r = nullptr;
  const double *a = nullptr;
  dhop_fuse fuse(bool sum) const
  {
    dhop_fuse f;
    f.skip = skip;
    f.skip_at = skip_at;
    if (sum) {
      f.partial = partial;
      f.resid = r;
      f.resid_a = a;
    }
    return f;
  }
};

int hop(const gbx_gauge_s *u, const dhop_cfg &cfg, gbx_spinor_s *out, const gbx_spinor_s *in, int dag, double alpha,
        double beta, const gbx_spinor_s *c, hipStream_t st, const dhop_fuse &f = dhop_fuse())
{
  return dhop_launch(u, out, in, dag, cfg, alpha, beta, c, st, false, SlotRange(), &f);
}

// out = Mooee^-1 Dhop in (dag: the adjoints), in one kernel where the launch
// shape holds whole columns of slices.
int mooee_inv_dhop(const gbx_gauge_s *u, const dhop_cfg &cfg, gbx_spinor_s *out, const gbx_spinor_s *in,
                   const gbx_dwf_params *dwf, int dag, hipStream_t st, dhop_fuse f)
{
  if (dhop_s5inv_fits(in, cfg)) {
    f.s5 = dhop_fuse::MOOEE_INV;
    f.dwf = dwf;
    return hop(u, cfg, out, in, dag, 0.0, 1.0, nullptr, st, f);
  }
  GBX_TRY(hop(u, cfg, out, in, dag, 0.0, 1.0, nullptr, st, f));
  return dwf_s5_launch(out, out, nullptr, dwf, 1, dag, 1.0, 0.0, st);
}

// out = Mooee c + beta Dhop in (dag: the adjoints) in one kernel.
int mooee_plus_dhop(const gbx_gauge_s *u, const dhop_cfg &cfg, gbx_spinor_s *out, const gbx_spinor_s *c,
                    const gbx_spinor_s *in, const gbx_dwf_params *dwf, int dag, double beta, hipStream_t st,
                    dhop_fuse f = dhop_fuse())
{
  f.s5 = dhop_fuse::MOOEE;
  f.dwf = dwf;
  return hop(u, cfg, out, in, dag, 1.0, beta, c, st, f);
}

// y = Mpc x (dag = 0) or Mpc^dag x (dag = 1), with dagger kernels for dag
// ((DhopEO DhopOE)^dag = (Dhop^dag)_EO (Dhop^dag)_OE):
//   Wilson:  to = DhopOE x;  y = x - kappa^2 DhopEO to
//   DWF:     to = Mooee^-1 DhopOE x;  y = Mooee x - DhopEO to / 4
int apply_schur(const NormalOp &op, gbx_spinor_s *y, const gbx_spinor_s *x, int dag, hipStream_t st,
                const Step &step = Step())
{
  if (op.kind == OP_DWF) {
    GBX_TRY(mooee_inv_dhop(op.uo, op.co, op.to, x, &op.dwf, dag, st, step.fuse(false)));
    return mooee_plus_dhop(op.ue, op.ce, y, x, op.to, &op.dwf, dag, -0.25, st, step.fuse(true));
  }
  GBX_TRY(hop(op.uo, op.co, op.to, x, dag, 0.0, 1.0, nullptr, st, step.fuse(false)));
  return hop(op.ue, op.ce, y, op.to, dag, 1.0, -op.kappa * op.kappa, x, st, step.fuse(true));
}

// y = M x or M^dag x on the whole lattice, x - kappa Dhop x.
int apply_m(const NormalOp &op, gbx_spinor_s *y, const gbx_spinor_s *x, int dag, hipStream_t st, const Step &step = Step())
{
  if (op.eo) return apply_schur(op, y, x, dag, st, step);
  return hop(op.ue, op.ce, y, x, dag, 1.0, -op.kappa, x, st, step.fuse(true));
}

// y = A x by way of t.
int apply_normal(const NormalOp &op, gbx_spinor_s *y, const gbx_spinor_s *x, hipStream_t st)
{
  GBX_TRY(apply_m(op, op.t, x, 0, st));
  return apply_m(op, y, op.t, 1, st);
}

// Partial sums an application leaves in Step::partial.
uint32_t normal_partials(const NormalOp &op) { return dhop_workgroups(op.ue, op.t, op.ce); }

// Waits until the device has reported iteration `seen` + 1 of the inner solve.
int next_word(const HostWords *h, uint32_t seen, hipStream_t st, uint64_t *word)
{
  for (uint32_t spin = 1;; spin++) {
    const uint64_t v = __atomic_load_n(&h->word, __ATOMIC_ACQUIRE);
    if ((uint32_t)v > seen) {
      *word = v;
      return GBX_OK;
    }
    if (spin % 4096 == 0) {  // everything enqueued has run and said nothing, or the device failed
      const hipError_t q = hipStreamQuery(st);
      if (q == hipSuccess && (uint32_t)__atomic_load_n(&h->word, __ATOMIC_ACQUIRE) <= seen)
        return gbx_fail(GBX_EHIP, "cg: the inner solve stopped reporting");
      if (q != hipSuccess && q != hipErrorNotReady)
        return gbx_fail(GBX_EHIP, "cg: the inner solve failed: %s", hipGetErrorString(q));
    }
    __builtin_ia32_pause();
  }
}

// Inner CG on A e = scale * src (src FP64): e, r in precision PE; p, its other
// buffer p2 and the operator's temporaries in PP (the gauge field's).  *it_out
// iterations ran; e is not written if that is 0.
template <int PE, int PP>
int inner_cg(const NormalOp &op, gbx_spinor_s *e, gbx_spinor_s *r, gbx_spinor_s *p, gbx_spinor_s *p2, const gbx_spinor_s *src,
             double scale, double rel_tol, int max_iter, uint32_t *it_out, int *applies, Scratch &sc, hipStream_t st)
{
  constexpr uint32_t kAhead = 3;  // iterations enqueued beyond the last one reported
  const uint64_t npts = r->geom->vol * (uint64_t)r->M;
  const int nb = blocks_for(npts);
  const int np = (int)normal_partials(op);
  const dim3 grid((unsigned)nb), block(kRT);
  HostWords *h = sc.host;
  __atomic_store_n(&h->word, 0ull, __ATOMIC_RELEASE);
  hipLaunchKernelGGL((k_cg_start<PE, PP>), grid, block, 0, st, scale, src->d, r->d, p->d, npts, r->M, sc.partial);
  hipLaunchKernelGGL(k_cg_begin, dim3(1), block, 0, st, sc.scal, (const double *)sc.partial, nb, rel_tol);
  GBX_HIP(hipGetLastError());
  auto fold = [&](uint32_t it, const double *part, int *n) -> const double * {
    if (*n <= kPlain) return part;
    hipLaunchKernelGGL(k_cg_fold, dim3(kFold), block, 0, st, (const CgScal *)sc.scal, it, part, *n, sc.fold);
    *n = kFold;
    return sc.fold;
  };
  gbx_spinor_s *pp[2] = {p, p2};
  auto enqueue = [&](uint32_t it) -> int {
    gbx_spinor_s *pi = pp[it & 1], *pn = pp[~it & 1];
    Step step;
    step.skip = &sc.scal->done_at;
    step.skip_at = it;
    step.partial = sc.tt;
    GBX_TRY(apply_m(op, op.t, pi, 0, st, step));
    int n = np;
    const double *tt = fold(it, sc.tt, &n);
    hipLaunchKernelGGL(k_cg_alpha, dim3(1), dim3(kAT), 0, st, sc.scal, it, tt, n);
    step.skip = &sc.scal->hop_at;
    step.partial = sc.tt;
    step.r = r;
    step.a = &sc.scal->alpha[it & 1];
    GBX_TRY(apply_m(op, pn, op.t, 1, st, step));  // pn: not written
    n = np;
    const double *rp = fold(it, sc.tt, &n);
    const int first = it < 2, last = it + 1 == (uint32_t)max_iter;
    if (it & 1)
      hipLaunchKernelGGL((k_cg_ep<PE, PP, true>), grid, block, 0, st, sc.scal, it, rp, n, r->d, pi->d, pn->d, e->d, npts, r->M,
                         first, last, &h->word);
    else
      hipLaunchKernelGGL((k_cg_ep<PE, PP, false>), grid, block, 0, st, sc.scal, it, rp, n, r->d, pi->d, pn->d, e->d, npts, r->M,
                         first, last, &h->word);
    GBX_HIP(hipGetLastError());
    return GBX_OK;
  };
  uint32_t sent = 0, seen = 0;
  bool broke = false;
  while (seen < (uint32_t)max_iter) {
    while (sent < (uint32_t)max_iter && sent < seen + kAhead) GBX_TRY(enqueue(sent++));
    uint64_t w;
    GBX_TRY(next_word(h, seen, st, &w));
    seen = (uint32_t)w;
    if (w >> 33) broke = true;
    if (w >> 32) break;
  }
  *it_out = broke ? seen - 1 : seen;
  *applies += (int)seen;
  return GBX_OK;
}

int inner_dispatch(const NormalOp &op, gbx_spinor_s *e, gbx_spinor_s *r, gbx_spinor_s *p, gbx_spinor_s *p2,
                   const gbx_spinor_s *src, double scale, double tol, int maxit, uint32_t *it, int *applies, Scratch &sc,
                   hipStream_t st)
{
  if (e->prec == GBX_F64) return inner_cg<GBX_F64, GBX_F64>(op, e, r, p, p2, src, scale, tol, maxit, it, applies, sc, st);
  switch (p->prec) {
  case GBX_F32: return inner_cg<GBX_F32, GBX_F32>(op, e, r, p, p2, src, scale, tol, maxit, it, applies, sc, st);
  case GBX_F16: return inner_cg<GBX_F32, GBX_F16>(op, e, r, p, p2, src, scale, tol, maxit, it, applies, sc, st);
  default: return inner_cg<GBX_F32, GBX_BF16>(op, e, r, p, p2, src, scale, tol, maxit, it, applies, sc, st);
  }
}

// z = a x + b y and |z|^2 (waits for it).
int axpby_norm(double a, const gbx_spinor_s *x, double b, const gbx_spinor_s *y, gbx_spinor_s *z, double *n2, Scratch &sc,
               hipStream_t st)
{
  const uint64_t n = z->geom->vol * (uint64_t)z->M * 12;
  const int nb = blocks_for(n);
  hipLaunchKernelGGL(k_axpby_norm, dim3((unsigned)nb), dim3(kRT), 0, st, a, x->d, b, y->d, z->d, n, sc.partial);
  GBX_HIP(hipGetLastError());
  return sc.fetch(st, nb, n2);
}

int axpy_into_f64(double a, const gbx_spinor_s *e, gbx_spinor_s *x, hipStream_t st)
{
  const uint64_t npts = x->geom->vol * (uint64_t)x->M;
  switch (e->prec) {
  case GBX_F64: hipLaunchKernelGGL(k_axpy_into_f64<GBX_F64>, dim3(kRB), dim3(kRT), 0, st, a, e->d, x->d, npts, x->M); break;
  case GBX_F32: hipLaunchKernelGGL(k_axpy_into_f64<GBX_F32>, dim3(kRB), dim3(kRT), 0, st, a, e->d, x->d, npts, x->M); break;
  case GBX_F16: hipLaunchKernelGGL(k_axpy_into_f64<GBX_F16>, dim3(kRB), dim3(kRT), 0, st, a, e->d, x->d, npts, x->M); break;
  default: hipLaunchKernelGGL(k_axpy_into_f64<GBX_BF16>, dim3(kRB), dim3(kRT), 0, st, a, e->d, x->d, npts, x->M); break;
  }
  GBX_HIP(hipGetLastError());
  return GBX_OK;
}

int check_params(const gbx_cg_params *p)
{
  GBX_CHECK(std::fabs(p->kappa) < 0.125, GBX_EINVAL, "cg: |kappa| = %g must be < 1/8", p->kappa);
  GBX_CHECK(p->tol > 0 && p->inner_tol > 0 && p->inner_tol < 1 && p->max_outer >= 1 && p->max_inner >= 1, GBX_EINVAL,
            "cg: bad tolerances or iteration limits");
  return GBX_OK;
}

int check_args(const gbx_gauge_s *u_hi, const gbx_gauge_s *u_lo, const gbx_spinor_s *x, const gbx_spinor_s *b,
               const gbx_cg_params *p)
{
  GBX_CHECK(u_hi && x && b && p, GBX_ENULL, "cg: NULL argument");
  GBX_CHECK(u_hi->prec == GBX_F64, GBX_EINVAL, "cg: the outer gauge field must be FP64");
  GBX_CHECK(x->prec == GBX_F64 && b->prec == GBX_F64, GBX_EINVAL, "cg: x and b must be FP64");
  GBX_CHECK(x->nrhs == 1 && b->nrhs == 1, GBX_EINVAL, "cg: one right-hand side");
  GBX_CHECK(x->geom == u_hi->geom && b->geom == u_hi->geom && x->Ls == b->Ls, GBX_EMISMATCH, "cg: shapes differ");
  GBX_CHECK(x->d != b->d, GBX_EALIAS, "cg: x aliases b");
  if (u_lo) {
    GBX_CHECK(u_lo->geom == u_hi->geom, GBX_EMISMATCH, "cg: inner gauge field on another geometry");
    GBX_CHECK(u_lo->prec != GBX_F64, GBX_EINVAL, "cg: the inner gauge field must be FP32, FP16 or BF16");
  }
  GBX_CHECK(whole_lattice(u_hi->geom), GBX_EINVAL,
            "cg: gbx_cg_solve works on a whole lattice; use gbx_cg_solve_eo on a red-black pair");
  return check_params(p);
}

int solve(const gbx_gauge_s *u_hi, const gbx_gauge_s *u_lo, gbx_spinor_s *x, const gbx_spinor_s *b, const gbx_cg_params *prm,
          gbx_cg_stats *stats)
{
  GBX_TRY(check_args(u_hi, u_lo, x, b, prm));
  // TDIAG fields: the solve runs in that basis (S is orthogonal, so norms
  // and residuals are the chiral ones); FP64 or FP32 inner solves only.
  GBX_CHECK(x->basis == b->basis, GBX_EMISMATCH, "cg: x and b are in different spin bases");
  GBX_CHECK(b->basis == GBX_BASIS_CHIRAL || !u_lo || u_lo->prec == GBX_F32, GBX_EUNSUPPORTED,
            "cg: TDIAG fields need an FP64 or FP32 inner gauge field");
  const auto t0 = std::chrono::steady_clock::now();
  gbx_cg_stats st{};
  gbx_geom_s *g = u_hi->geom;
  hipStream_t s = g->stream;
  const int Ls = x->Ls;
  const int plo = u_lo ? u_lo->prec : GBX_F64;
  const int pe = u_lo ? GBX_F32 : GBX_F64;
  Workspace w;
  gbx_spinor_s r, t, y, e, ri, p, p2, tl;
  for (gbx_spinor_s *f : {&r, &t, &y}) w.field(*f, g, Ls, GBX_F64, b->basis);
  for (gbx_spinor_s *f : {&e, &ri}) w.field(*f, g, Ls, pe, b->basis);
  for (gbx_spinor_s *f : {&p, &p2, &tl}) w.field(*f, g, Ls, plo, b->basis);
  NormalOp op_hi{false, u_hi, nullptr, prm->kappa, &t, nullptr};
  NormalOp op_lo{false, u_lo ? u_lo : u_hi, nullptr, prm->kappa, &tl, nullptr};
  op_hi.shapes();
  op_lo.shapes();
  Scratch sc;
  sc.plan(w, normal_partials(op_lo));
  GBX_TRY(w.allocate(s));
  GBX_TRY(sc.init(w));
  double bb;
  GBX_TRY(spinor_norm2_on(b, &bb, s));
  GBX_CHECK(bb > 0.0, GBX_EINVAL, "cg: b is zero");
  const double bnorm = std::sqrt(bb);
  const double N = (double)g->vol * Ls * 24;
  double rel = 1.0;
  for (;;) {
    // true residual r = b - M^dag M x in FP64
    GBX_TRY(apply_normal(op_hi, &y, x, s));
    st.hi_applies++;
    double rr;
    GBX_TRY(axpby_norm(1.0, b, -1.0, &y, &r, &rr, sc, s));
    rel = std::sqrt(rr) / bnorm;
    if (rel <= prm->tol || st.outer_iters >= prm->max_outer || !(rr > 0.0)) break;
    const double scale = std::sqrt(N) / std::sqrt(rr);
    uint32_t it = 0;
    GBX_TRY(inner_dispatch(op_lo, &e, &ri, &p, &p2, &r, scale, prm->inner_tol, prm->max_inner, &it, &st.lo_applies, sc, s));
    if (it) GBX_TRY(axpy_into_f64(1.0 / scale, &e, x, s));
    st.inner_iters += (int)it;
    st.outer_iters++;
  }
  GBX_HIP(hipStreamSynchronize(s));
  st.true_resid = rel;
  st.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  if (stats) *stats = st;
  if (rel > prm->tol) return gbx_fail(GBX_ENOCONV, "cg: relative residual %.3e after %d outer iterations", rel, st.outer_iters);
  return GBX_OK;
}

// Even-odd Schur-complement solve on a red-black pair (kind = OP_WILSON:
// M = 1 - kappa Dhop; OP_DWF: D = Mooee - Dhop / 2).
int solve_schur(int kind, const gbx_dwf_params *dwf, const gbx_gauge_s *const u_hi[2], const gbx_gauge_s *const *u_lo,
                gbx_spinor_s *const x[2], const gbx_spinor_s *const b[2], const gbx_cg_params *prm, gbx_cg_stats *stats)
{
  const char *who = kind == OP_DWF ? "dwf_eo" : "cg_eo";
  GBX_CHECK(u_hi && x && b && prm && u_hi[0] && u_hi[1] && x[0] && x[1] && b[0] && b[1], GBX_ENULL, "%s: NULL argument", who);
  const gbx_geom_s *ge = u_hi[0]->geom, *go = u_hi[1]->geom;
  GBX_CHECK(ge->parity == 0 && go->parity == 1 && ge->pair_id == go->pair_id, GBX_EMISMATCH,
            "%s: u_hi must be the even then the odd half of one red-black pair", who);
  GBX_CHECK(ge->nghost == 0, GBX_EINVAL, "%s: the solvers take a whole lattice's halves, not a domain part's", who);
  const int basis = b[0]->basis;
  GBX_CHECK(x[0]->basis == basis && x[1]->basis == basis && b[1]->basis == basis, GBX_EMISMATCH,
            "%s: x and b are in different spin bases", who);
  for (int p = 0; p < 2; p++) {
    const gbx_geom_s *g = p ? go : ge;
    GBX_CHECK(u_hi[p]->prec == GBX_F64, GBX_EINVAL, "%s: the outer gauge fields must be FP64", who);
    GBX_CHECK(x[p]->prec == GBX_F64 && b[p]->prec == GBX_F64, GBX_EINVAL, "%s: x and b must be FP64", who);
    GBX_CHECK(x[p]->geom == g && b[p]->geom == g, GBX_EMISMATCH, "%s: x[%d] / b[%d] not on the %s half", who, p, p,
              p ? "odd" : "even");
    GBX_CHECK(x[p]->nrhs == 1 && b[p]->nrhs == 1 && x[p]->Ls == x[0]->Ls && b[p]->Ls == x[0]->Ls, GBX_EMISMATCH,
              "%s: one right-hand side, equal Ls", who);
    GBX_CHECK(x[p]->d != b[p]->d, GBX_EALIAS, "%s: x aliases b", who);
    if (u_lo) {
      GBX_CHECK(u_lo[p] && u_lo[p]->geom == g, GBX_EMISMATCH, "%s: inner gauge field %d not on the %s half", who, p,
                p ? "odd" : "even");
      GBX_CHECK(u_lo[p]->prec != GBX_F64 && u_lo[p]->prec == u_lo[0]->prec, GBX_EINVAL,
                "%s: inner gauge fields must share one of FP32, FP16, BF16", who);
    }
  }
  // TDIAG fields: the Wilson operator only (the DWF terms' chirality
  // projectors are written for chiral values), FP64 or FP32 inner solves.
  GBX_CHECK(basis == GBX_BASIS_CHIRAL || (kind == OP_WILSON && (!u_lo || u_lo[0]->prec == GBX_F32)), GBX_EUNSUPPORTED,
            "%s: TDIAG fields: the Wilson operator with an FP64 or FP32 inner solve only", who);
  if (kind == OP_DWF) {
    GBX_CHECK(prm->tol > 0 && prm->inner_tol > 0 && prm->inner_tol < 1 && prm->max_outer >= 1 && prm->max_inner >= 1,
              GBX_EINVAL, "%s: bad tolerances or iteration limits", who);
  } else {
    GBX_TRY(check_params(prm));
  }
  const auto t0 = std::chrono::steady_clock::now();
  gbx_cg_stats st{};
  gbx_geom_s *g = u_hi[0]->geom, *g1 = u_hi[1]->geom;
  hipStream_t s = g->stream;  // the pair's one stream
  const int Ls = x[0]->Ls;
  const double kappa = prm->kappa;
  const int plo = u_lo ? u_lo[0]->prec : GBX_F64;
  const int pe = u_lo ? GBX_F32 : GBX_F64;
  Workspace w;
  gbx_spinor_s bp, r, y, t, to, e, ri, p, p2, tl, tol_, ro;
  for (gbx_spinor_s *f : {&bp, &r, &y, &t}) w.field(*f, g, Ls, GBX_F64, basis);
  for (gbx_spinor_s *f : {&to, &ro}) w.field(*f, g1, Ls, GBX_F64, basis);
  for (gbx_spinor_s *f : {&e, &ri}) w.field(*f, g, Ls, pe, basis);
  for (gbx_spinor_s *f : {&p, &p2, &tl}) w.field(*f, g, Ls, plo, basis);
  w.field(tol_, g1, Ls, plo, basis);
  NormalOp op_hi{true, u_hi[0], u_hi[1], kappa, &t, &to};
  NormalOp op_lo{true, u_lo ? u_lo[0] : u_hi[0], u_lo ? u_lo[1] : u_hi[1], kappa, &tl, &tol_};
  op_hi.kind = op_lo.kind = kind;
  if (kind == OP_DWF) op_hi.dwf = op_lo.dwf = *dwf;
  op_hi.shapes();
  op_lo.shapes();
  Scratch sc;
  sc.plan(w, normal_partials(op_lo));
  GBX_TRY(w.allocate(s));
  GBX_TRY(sc.init(w));
  double bbe, bbo;
  GBX_TRY(spinor_norm2_on(b[0], &bbe, s));
  GBX_TRY(spinor_norm2_on(b[1], &bbo, s));
  GBX_CHECK(bbe + bbo > 0.0, GBX_EINVAL, "%s: b is zero", who);
  const double bnorm = std::sqrt(bbe + bbo);
  const double N = (double)g->vol * Ls * 24;
  // b'_e:  Wilson b_e + kappa DhopEO b_o;  DWF b_e + DhopEO Mooee^-1 b_o / 2
  if (kind == OP_DWF) {
    GBX_TRY(dwf_s5_launch(&to, b[1], nullptr, dwf, 1, 0, 1.0, 0.0, s));
    GBX_TRY(hop(u_hi[0], op_hi.ce, &bp, &to, 0, 1.0, 0.5, b[0], s));
  } else {
    GBX_TRY(hop(u_hi[0], op_hi.ce, &bp, b[1], 0, 1.0, kappa, b[0], s));
  }
  double rel = 1.0;
  for (;;) {
    // r = b'_e - Mpc x_e in FP64; |r| is |b - M x| once x_o is rebuilt
    GBX_TRY(apply_schur(op_hi, &y, x[0], 0, s));
    st.hi_applies++;
    double rr;
    GBX_TRY(axpby_norm(1.0, &bp, -1.0, &y, &r, &rr, sc, s));
    rel = std::sqrt(rr) / bnorm;
    if (rel <= prm->tol || st.outer_iters >= prm->max_outer || !(rr > 0.0)) break;
    // inner right-hand side Mpc^dag r, scaled to unit-RMS entries
    GBX_TRY(apply_schur(op_hi, &y, &r, 1, s));
    double yy;
    GBX_TRY(spinor_norm2_on(&y, &yy, s));
    if (!(yy > 0.0)) break;
    const double scale = std::sqrt(N) / std::sqrt(yy);
    uint32_t it = 0;
    GBX_TRY(inner_dispatch(op_lo, &e, &ri, &p, &p2, &y, scale, prm->inner_tol, prm->max_inner, &it, &st.lo_applies, sc, s));
    if (it) GBX_TRY(axpy_into_f64(1.0 / scale, &e, x[0], s));
    st.inner_iters += (int)it;
    st.outer_iters++;
  }
  if (kind == OP_DWF) {
    // x_o = Mooee^-1 (b_o + DhopOE x_e / 2); then b - D x with D = Mooee - Dhop / 2
    GBX_TRY(hop(u_hi[1], op_hi.co, &to, x[0], 0, 1.0, 0.5, b[1], s));
    GBX_TRY(dwf_s5_launch(x[1], &to, nullptr, dwf, 1, 0, 1.0, 0.0, s));
    GBX_TRY(mooee_plus_dhop(u_hi[0], op_hi.ce, &y, x[0], x[1], dwf, 0, -0.5, s));   // (D x)_e
    GBX_TRY(mooee_plus_dhop(u_hi[1], op_hi.co, &to, x[1], x[0], dwf, 0, -0.5, s));  // (D x)_o
  } else {
    // x_o = b_o + kappa DhopOE x_e; then b - M x
    GBX_TRY(hop(u_hi[1], op_hi.co, x[1], x[0], 0, 1.0, kappa, b[1], s));
    GBX_TRY(hop(u_hi[0], op_hi.ce, &y, x[1], 0, 1.0, -kappa, x[0], s));   // (M x)_e
    GBX_TRY(hop(u_hi[1], op_hi.co, &to, x[0], 0, 1.0, -kappa, x[1], s));  // (M x)_o
  }
  double re2, ro2;
  GBX_TRY(axpby_norm(1.0, b[0], -1.0, &y, &r, &re2, sc, s));
  GBX_TRY(axpby_norm(1.0, b[1], -1.0, &to, &ro, &ro2, sc, s));
  GBX_HIP(hipStreamSynchronize(s));
  const double full = std::sqrt(re2 + ro2) / bnorm;
  st.true_resid = full;
  st.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  if (stats) *stats = st;
  if (rel > prm->tol)
    return gbx_fail(GBX_ENOCONV, "%s: relative residual %.3e after %d outer iterations", who, rel, st.outer_iters);
  return GBX_OK;
}

}  // namespace

extern "C" int gbx_cg_solve_eo(const gbx_gauge u_hi[2], const gbx_gauge *u_lo, gbx_spinor x[2], const gbx_spinor b[2],
                               const gbx_cg_params *p, gbx_cg_stats *st)
{
  return solve_schur(OP_WILSON, nullptr, u_hi, u_lo, x, b, p, st);
}

extern "C" int gbx_dwf_solve_eo(const gbx_gauge u_hi[2], const gbx_gauge *u_lo, gbx_spinor x[2], const gbx_spinor b[2],
                                const gbx_dwf_params *dwf, const gbx_cg_params *p, gbx_cg_stats *st)
{
  GBX_CHECK(dwf, GBX_ENULL, "dwf_eo: NULL DWF parameters");
  GBX_CHECK(x && x[0], GBX_ENULL, "dwf_eo: NULL argument");
  GBX_CHECK(5.0 - dwf->M5 > 0.0 && x[0]->Ls >= 2 && x[0]->Ls <= 256, GBX_EINVAL, "dwf_eo: M5 = %g, Ls = %d", dwf->M5,
            x[0]->Ls);
  return solve_schur(OP_DWF, dwf, u_hi, u_lo, x, b, p, st);
}

extern "C" int gbx_cg_solve(gbx_gauge u_hi, gbx_gauge u_lo, gbx_spinor x, gbx_spinor b, const gbx_cg_params *p,
                            gbx_cg_stats *st)
{
  GBX_CHECK(u_lo, GBX_ENULL, "gbx_cg_solve: NULL inner gauge field (use gbx_cg_solve_f64)");
  return solve(u_hi, u_lo, x, b, p, st);
}

extern "C" int gbx_cg_solve_f64(gbx_gauge u, gbx_spinor x, gbx_spinor b, const gbx_cg_params *p, gbx_cg_stats *st)
{
  return solve(u, nullptr, x, b, p, st);
}
