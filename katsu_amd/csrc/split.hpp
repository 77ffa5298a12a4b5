// split.hpp -- what the C ABI (katsu_hip.hip) calls of the split-bf16 kernels,
// which are compiled apart from it (split.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace katsu {

// One product C[M,N] = beta*C + op(A) op(B); row-major, packed.
struct SplitProblem {
    const float *a, *b;
    float *c;
    int64_t M, N, K;
    int ta, tb;
    float beta;
};

// Whether split_gemm takes p: operands below 1 GiB, the output below 2^31.
bool split_gemm_ok(const SplitProblem &p);
// Launches p; a katsu_status.
int split_gemm(const SplitProblem &p, hipStream_t st);
// Both, p with ta = 0, tb = 1 and q with ta = 1, tb = 0: in one launch unless two
// are estimated to take less.
int split_gemm_vjp(const SplitProblem &p, const SplitProblem &q, hipStream_t st);

// A convolution layer: x [N][C][H][W], w [K][C][R][S], stride st, padding pad.
struct SplitLayer {
    int N, C, H, W, K, R, S, st, pad, OH, OW;
};

// The forward pass and the data gradient, dx = beta*dx + dX.  below: the time
// the float32 kernels would take, in microseconds.  kLaunched: *rc is the
// launch's katsu_status; kSlower: not in less than that time; kUnfit: not a layer
// these kernels take.
enum class SplitRun { kLaunched, kSlower, kUnfit };
SplitRun split_conv_fwd(const float *x, const float *w, float *y, const SplitLayer &l,
                        double below, hipStream_t st, int *rc);
SplitRun split_conv_dx(const float *gy, const float *w, float *dx, const SplitLayer &l, float beta,
                       double below, hipStream_t st, int *rc);

// The filter gradient, dw = beta*dw + dW.  split_dw_bytes: the workspace it
// needs, 0 if it does not take the layer.
size_t split_dw_bytes(const SplitLayer &l);
int split_dw(const float *x, const float *gy, float *dw, const SplitLayer &l, float beta, float *ws,
             hipStream_t st);

}  // namespace katsu
