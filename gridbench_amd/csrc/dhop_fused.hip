// Instantiations of the hopping kernel (dhop_kernel.h) that carry more of a
// solver's operator in their epilogue: the domain-wall fifth-dimension terms,
// and |out|^2 of the output they write.
//
// The hopping kernels are bound by their gathers (dhop.hip), so what an
// epilogue adds is the traffic of its own operands: D = Mooee - Dhop / 2 at
// 24^4 x Ls16 FP64 took 836 us for Dhop and 491 us for a pass over three
// fields that adds Mooee; in one kernel it takes 857 us (FP32: 627 -> 424 us),
// 50 us over Dhop alone for a third field to read.  The even-odd operator's
// Mooee^-1 DhopOE (16^4 x Ls12 FP32: 29 + 16 us as two kernels) saves the pass
// over the half lattice too; the domain-wall solve there went from 26.4 to
// 22.2 ms with both.
#include "dhop_kernel.h"

namespace dhopk {

namespace {

template <int P, bool DAG, bool C12, int EPI, bool TD, int RED>
void pick_pf(int pf, const LaunchArgs &a)
{
  if (pf) launch_t<P, DAG, C12, EPI, 1, false, false, TD, RED>(a);
  else launch_t<P, DAG, C12, EPI, 0, false, false, TD, RED>(a);
}

template <int P, bool C12, int EPI, bool TD = false>
void pick_red(bool dag, int red, int pf, const LaunchArgs &a)
{
  if (dag) {
    if (red) pick_pf<P, true, C12, EPI, TD, RED_RESID>(pf, a);
    else pick_pf<P, true, C12, EPI, TD, RED_NONE>(pf, a);
  } else {
    if (red) pick_pf<P, false, C12, EPI, TD, RED_OUT>(pf, a);
    else pick_pf<P, false, C12, EPI, TD, RED_NONE>(pf, a);
  }
}

template <int P, bool C12>
void pick_epi(int epi, bool dag, bool td, int red, int pf, const LaunchArgs &a)
{
  if (epi == EPI_S5INV) {
    if (dag) pick_pf<P, true, C12, EPI_S5INV, false, RED_NONE>(pf, a);
    else pick_pf<P, false, C12, EPI_S5INV, false, RED_NONE>(pf, a);
  } else if (epi == EPI_S5) {
    pick_red<P, C12, EPI_S5>(dag, red, pf, a);
  } else if (epi == EPI_S5X) {
    pick_red<P, C12, EPI_S5X>(dag, red, pf, a);
  } else {
    if constexpr (P == GBX_F64 || P == GBX_F32) {
      if (td) {
        if (dag) pick_pf<P, true, C12, EPI_AXPBY, true, RED_RESID>(pf, a);
        else pick_pf<P, false, C12, EPI_AXPBY, true, RED_OUT>(pf, a);
        return;
      }
    }
    if (dag) pick_pf<P, true, C12, EPI_AXPBY, false, RED_RESID>(pf, a);
    else pick_pf<P, false, C12, EPI_AXPBY, false, RED_OUT>(pf, a);
  }
}

template <int P>
void pick_c12(int epi, bool dag, bool c12, bool td, int red, int pf, const LaunchArgs &a)
{
  if (c12) pick_epi<P, true>(epi, dag, td, red, pf, a);
  else pick_epi<P, false>(epi, dag, td, red, pf, a);
}

}  // namespace

void launch_fused(int prec, int epi, bool dag, bool c12, bool td, int red, int pf, const LaunchArgs &a)
{
  switch (prec) {
  case GBX_F64: pick_c12<GBX_F64>(epi, dag, c12, td, red, pf, a); break;
  case GBX_F32: pick_c12<GBX_F32>(epi, dag, c12, td, red, pf, a); break;
  case GBX_F16: pick_c12<GBX_F16>(epi, dag, c12, td, red, pf, a); break;
  default: pick_c12<GBX_BF16>(epi, dag, c12, td, red, pf, a); break;
  }
}

}  // namespace dhopk
