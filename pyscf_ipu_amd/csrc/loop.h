// Forms of the public entry points that the native SCF loop (rks.hip) chains
// with fewer launches: outputs that a kernel of the sequence has already zeroed,
// zeroing of a later kernel's output on the side, results written straight to
// pinned host memory.  Arguments are checked by the callers.
#pragma once
#include "common.h"

namespace pscf {

// pscf_scf_step; afterwards zero_v[N * N] and *zero_e are 0 (if not null; zero_v
// may be the Vxc that the step reads).
int scf_step_zero(int dtype, int iteration, int N, int nocc, const double* d_Hcore, const double* d_S,
                  const double* d_Linv, const void* d_dJK, const void* d_Vxc, double* d_D, double* d_H,
                  double* d_mo_energy, double* d_C, void* d_state, int use_diis, double* zero_v, double* zero_e,
                  hipStream_t st);

// pscf_energy; host (a device address of pinned memory, or null) also receives
// the five terms and mo_e[N].
int energy_to_host(int dtype, int N, const double* d_D, const double* d_Hcore, const void* d_dJK, const double* d_exc,
                   double e_nuc, double* d_out, const double* mo_e, double* host, hipStream_t st);

// pscf_xc in FP64; zeroed: exc and vxc already hold 0; zero[nzero] is set to 0.
int xc_f64(const double* ao, int64_t sc, int64_t smu, int64_t sp, int g, int N, const double* dm, const double* w,
           double eps, double* exc, double* vxc, void* ws, size_t ws_bytes, bool zeroed, double* zero, int64_t nzero,
           hipStream_t st);

// pscf_jk_s8 in FP64 into an out that already holds 0.
int jk_s8_f64_zeroed(const double* eri, int N, const double* dm, double hyb, double* out, void* ws, size_t ws_bytes,
                     hipStream_t st);

}  // namespace pscf
