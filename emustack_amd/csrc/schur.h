// Schur form of complex upper Hessenberg matrices on the host.
#pragma once
#include <complex>

namespace emu {
// whether this CPU has the vector instructions that these are written in
bool schur_available();
// A (n x n, column-major) <- Q^H A Q upper Hessenberg, Q (n x n) overwritten.
void schur_reduce(int n, std::complex<double> *A, int lda, std::complex<double> *Q, int ldq);
// H (n x n, upper Hessenberg, column-major) <- T = W^H H W upper triangular,
// Z (nz x n) <- Z W.  False when an iteration limit was reached (H and Z are
// then some unitary similarity of the input, not yet triangular).
bool schur_hessenberg(int n, std::complex<double> *H, int ldh, std::complex<double> *Z, int ldz, int nz);
// The rows of the upper triangular T (n x n) with sel[i] != 0 to the top, in
// their order, by a unitary similarity W: T <- W^H T W, Z (nz x n) <- Z W.
void schur_reorder(int n, std::complex<double> *T, int ldt, std::complex<double> *Z, int ldz, int nz, const int *sel);
}  // namespace emu
