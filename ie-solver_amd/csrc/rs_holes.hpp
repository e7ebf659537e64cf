// Launch wrappers for the bordered (multiply connected) system.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "rs_device.hpp"

namespace iegpu {

void launch_mark_skel(const DevState& s, int* mask, int64_t ndof,
                      hipStream_t st);
void launch_copy(double* dst, const double* src, int64_t n, hipStream_t st);
// Row gather: dst row r = src row map[r] (rows of row_words 32-bit words;
// map[r] < 0 zeroes the row).  Every map entry indexes a row of src.
void launch_gather_rows(void* dst, const void* src, const int* map, int n_rows, int row_words,
                        hipStream_t st);
// The border blocks U, Psi^T and their swept forms are row-major, ndof x h.
// partial holds border_partials(ndof, h) doubles.
int64_t border_partials(int64_t ndof, int h);
void launch_border_gram(const double* P, const double* C, const int* mask,
                        int64_t ndof, int h, double* partial, double* out,
                        hipStream_t st);
// S into Smat (destroyed) and its inverse into Sinv ((ncap + h)^2 doubles
// each); Spiv: ncap + h + kInvFlags ints.
template <typename R>
void launch_border_factor(const DevState& s, const double* mU, const double* mPsiT,
                          const double* gram, int h, double* Smat, double* Sinv, int* Spiv,
                          hipStream_t st);
// [x(skel); alpha] = S^{-1} [x(skel); g - mPsi^T(red,:) x(red)]; rhs:
// ncap + h doubles.
void launch_border_solve(const DevState& s, const double* mPsiT, const double* Sinv,
                         const int* mask, int64_t ndof, int h, double* x, const double* g,
                         double* alpha, double* partial, double* rhs, hipStream_t st);
void launch_red_update(double* x, const double* C, const int* mask,
                       const double* alpha, int64_t ndof, int h,
                       hipStream_t st);
// Border of the multiply connected operator: y += U alpha; z = Psi x - alpha.
void launch_border_apply(const double* U, const double* PsiT, const double* x,
                         const double* alpha, int64_t ndof, int h, double* partial, double* y,
                         double* z, hipStream_t st);

}  // namespace iegpu
