// The preconditioned flexible BiCGSTAB solves of km_twolevel.hip as one
// launch (km_persist.hip), for systems that fit the GPU's registers.
// Internal; not part of the C-ABI.
#pragma once

#include "km_common.h"

struct km_coarse;

namespace kmpersist {

// Whether a two-level solve of an NX x NY system on level C, or a smoothed
// solve of one, runs in one launch on this device; its tile shape in *shape.
bool fits_twolevel(km_ctx* ctx, const km_coarse* C, int NX, int NY, int* shape);
bool fits_smooth(km_ctx* ctx, int NX, int NY, int* shape);

// Inner flexible BiCGSTAB for A d = rhs from d = 0, results as
// kmcoarse::fused_inner (two-level preconditioner on ctx->coarse) and
// kmcoarse::smooth_inner / smooth_inner2 (red-black Gauss-Seidel sweeps).  ws:
// 2 n values of T (of each system).  coef: FP64 planes for the two-level
// solve, planes of T for the smoothed one.  *ran = false: the launch gave up
// before its end (a boundary row that couples to the interior, or a wait that
// ran into its time limit) and the caller takes its other path.
template <typename T>
int twolevel(km_ctx* ctx, int shape, int NX, int NY, const double* coef, const T* rhs, T* xd, T* ws, double eps,
             int max_iter, KState* out, const std::function<int()>* tail, bool* ran);
template <typename T>
int smooth(km_ctx* ctx, int nsys, const int* NX, const int* NY, const T* const* coef, const T* const* rhs,
           T* const* xd, T* const* ws, double eps, const int* max_iter, int sweeps, KState* out,
           const std::function<int()>* tail, bool* ran);

// What orders these launches on one device; created with the first context there.
int gate(int device);

// Plain BiCGSTAB, or CG, of a system whose first residual is rin (from_x: x
// holds x0, else x = 0 and rin = b), relative to ref = ||b||^2 (0: to ||rin||^2),
// as bicgstab_typed / cg_typed of km_krylov.hip.  ws: 2 n values.  words: null,
// or plain_words_bytes() of the caller's for the exchange.
bool fits_plain(km_ctx* ctx, int NX, int NY, int* shape);
size_t plain_words_bytes();
int plain(km_ctx* ctx, int shape, bool cg, int NX, int NY, const double* coef, const double* rin, double* x, bool from_x,
          double* ws, void* words, double eps, int max_iter, double ref, KState* out, const std::function<int()>* tail,
          bool* ran);

}  // namespace kmpersist

void km_persist_free(km_ctx* ctx);
