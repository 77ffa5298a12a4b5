// split.hip -- launches of the kernels that run float32 products on the bf16
// matrix cores (split3.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/katsu_hip.h"
#include "split.hpp"
#include "splitgemm.hpp"

namespace katsu {
namespace {

constexpr int64_t kMaxElems = (int64_t)1 << 28;  // 1 GiB of floats
constexpr int kCUs = 256;

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Blocks are dispatched round-robin over the 8 XCDs: each XCD gets a run of
// neighbouring tiles, whose operand panels its L2 then holds.
__device__ __forceinline__ int xcd_run(int b, int nb) {
    const int per = nb >> 3, rem = nb & 7;
    const int x = b & 7, idx = b >> 3;
    return x * per + (x < rem ? x : rem) + idx;
}

// The tiles.  T: side of the output tile (256: 256 x 128).
template <int T, bool TA, bool TB>
struct Tile;
template <bool TA, bool TB>
struct Tile<256, TA, TB> : SplitGemm<256, 128, 32, 64, 64, TA, TB> {};
template <bool TA, bool TB>
struct Tile<128, TA, TB> : SplitGemm<128, 128, 32, 64, 64, TA, TB> {};
template <bool TA, bool TB>
struct Tile<64, TA, TB> : SplitGemmRd<64, 64, 8, TA, TB> {};
template <bool TA, bool TB>
struct Tile<32, TA, TB> : SplitGemmRd<32, 32, 8, TA, TB> {};

template <int T>
constexpr int kThreadsOf = Tile<T, false, false>::kThreads;
// Waves per SIMD the registers allow: one for the 128-tile, two for the others.
template <int T>
constexpr int kOcc = T == 128 ? 1 : 2;

template <int T, bool TA, bool TB>
__global__ void __launch_bounds__(kThreadsOf<T>, kOcc<T>) split_gemm_kernel(const SplitGemmArgs g) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    Tile<T, TA, TB>::run(g, xcd_run(blockIdx.x, gridDim.x), lds);
}

// The first nb0 blocks do p (A B^T), the others q (A^T B).
template <int T>
__global__ void __launch_bounds__(kThreadsOf<T>, kOcc<T>)
    split_gemm_vjp_kernel(const SplitGemmArgs p, const SplitGemmArgs q, int nb0) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int b = blockIdx.x;
    if (b < nb0)
        Tile<T, false, true>::run(p, xcd_run(b, nb0), lds);
    else
        Tile<T, true, false>::run(q, xcd_run(b - nb0, gridDim.x - nb0), lds);
}

int status_of(hipError_t e) {
    if (e == hipSuccess) return KATSU_OK;
    return e == hipErrorNoDevice || e == hipErrorInvalidDevice ? KATSU_E_NODEVICE : KATSU_E_LAUNCH;
}

// Dynamic LDS above 64 KiB must be opted into, once per kernel function.
template <auto Kern>
int lds_optin(size_t bytes) {
    if (bytes <= 65536) return KATSU_OK;
    static const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void *>(Kern),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    return status_of(e);
}

SplitGemmArgs args_of(const SplitProblem &p, int T) {
    SplitGemmArgs g{};
    g.a = p.a;
    g.b = p.b;
    g.c = p.c;
    g.M = (int)p.M;
    g.N = (int)p.N;
    g.K = (int)p.K;
    g.lda = (int)(p.ta ? p.M : p.K);
    g.ldb = (int)(p.tb ? p.K : p.N);
    g.ldc = (int)p.N;
    g.a_bytes = (uint32_t)(p.M * p.K * 4);
    g.b_bytes = (uint32_t)(p.K * p.N * 4);
    g.beta = p.beta;
    g.tiles_m = (int)cdiv(p.M, T);
    g.tiles_n = (int)cdiv(p.N, T == 256 ? 128 : T);
    g.group = 8;
    return g;
}

int64_t tiles_of(const SplitProblem &p, int T) {
    return cdiv(p.M, T) * cdiv(p.N, T == 256 ? 128 : T);
}

// The tile of least estimated time, in ns: a round is one block on every CU,
// and costs a fixed part and a part per k.  Fitted to measured times: 256 x 128
// tiles 4096^3 in 627 us (2 rounds) and 4096 x 16 x 4096 in 24; 128-tiles
// 2048^3 in 111 us (1 round); 64-tiles 1024^3 in 20.4 us (1 round) and 2048^3
// in 126 (4); 32-tiles 300^3 in 6.2 us and 64 x 8192 x 64 in 50 (1 round each).
// The larger tiles read and split less per product, the smaller ones leave
// fewer CUs idle.
struct TileCost { int T; double fixed, per_k; };
constexpr TileCost kTileCost[] = {{256, 8000, 74}, {128, 5000, 51}, {64, 2000, 15}, {32, 1000, 6.5}};
constexpr double kLaunchNs = 3000;

double tile_ns(const TileCost &c, int64_t tiles, double k) {
    return kLaunchNs + (double)cdiv(tiles, kCUs) * (c.fixed + c.per_k * k);
}

int tile_for(const SplitProblem &p, double *ns) {
    int best = 0;
    for (const TileCost &c : kTileCost) {
        const double t = tile_ns(c, tiles_of(p, c.T), (double)p.K);
        if (!best || t < *ns) {
            best = c.T;
            *ns = t;
        }
    }
    return best;
}

// The tile for both products in one launch, or 0 where two launches are
// estimated to take less (products that want different tiles: 4096 x 4096 x 1
// with 98 us in one launch).
int tile_for_vjp(const SplitProblem &p, const SplitProblem &q) {
    double np, nq, one = 0;
    tile_for(p, &np);
    tile_for(q, &nq);
    int best = 0;
    for (const TileCost &c : kTileCost) {
        const int64_t tp = tiles_of(p, c.T), tq = tiles_of(q, c.T);
        const double k = ((double)tp * p.K + (double)tq * q.K) / (double)(tp + tq);
        // The longer sum of the two bounds a launch of few tiles.
        const double t =
            std::max(tile_ns(c, tp + tq, k), tile_ns(c, 1, (double)std::max(p.K, q.K)));
        if (!best || t < one) {
            best = c.T;
            one = t;
        }
    }
    return one < np + nq ? best : 0;
}

template <int T, bool TA, bool TB>
int launch(const SplitProblem &p, hipStream_t st) {
    constexpr auto kern = split_gemm_kernel<T, TA, TB>;
    const int rc = lds_optin<kern>(Tile<T, TA, TB>::kLds);
    if (rc != KATSU_OK) return rc;
    kern<<<dim3((unsigned)tiles_of(p, T)), dim3(kThreadsOf<T>), Tile<T, TA, TB>::kLds, st>>>(
        args_of(p, T));
    return status_of(hipGetLastError());
}

template <int T>
int launch_t(const SplitProblem &p, hipStream_t st) {
    if (p.ta) return p.tb ? launch<T, true, true>(p, st) : launch<T, true, false>(p, st);
    return p.tb ? launch<T, false, true>(p, st) : launch<T, false, false>(p, st);
}

template <int T>
int launch_vjp(const SplitProblem &p, const SplitProblem &q, hipStream_t st) {
    constexpr auto kern = split_gemm_vjp_kernel<T>;
    constexpr size_t lds = std::max(Tile<T, false, true>::kLds, Tile<T, true, false>::kLds);
    const int rc = lds_optin<kern>(lds);
    if (rc != KATSU_OK) return rc;
    const int64_t n0 = tiles_of(p, T), n1 = tiles_of(q, T);
    kern<<<dim3((unsigned)(n0 + n1)), dim3(kThreadsOf<T>), lds, st>>>(args_of(p, T), args_of(q, T),
                                                                     (int)n0);
    return status_of(hipGetLastError());
}

}  // namespace

bool split_gemm_ok(const SplitProblem &p) {
    return p.M * p.K < kMaxElems && p.K * p.N < kMaxElems && p.M * p.N < (int64_t)1 << 31;
}

int split_gemm(const SplitProblem &p, hipStream_t st) {
    double ns;
    switch (tile_for(p, &ns)) {
        case 256: return launch_t<256>(p, st);
        case 128: return launch_t<128>(p, st);
        case 64: return launch_t<64>(p, st);
        default: return launch_t<32>(p, st);
    }
}

int split_gemm_vjp(const SplitProblem &p, const SplitProblem &q, hipStream_t st) {
    switch (tile_for_vjp(p, q)) {
        case 0: {
            const int rc = split_gemm(p, st);
            return rc == KATSU_OK ? split_gemm(q, st) : rc;
        }
        case 256: return launch_vjp<256>(p, q, st);
        case 128: return launch_vjp<128>(p, q, st);
        case 64: return launch_vjp<64>(p, q, st);
        default: return launch_vjp<32>(p, q, st);
    }
}

}  // namespace katsu
