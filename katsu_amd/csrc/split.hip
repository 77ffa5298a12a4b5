// split.hip -- launches of the kernels that run float32 products on the bf16
// matrix cores (split3.hpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <utility>

#include "../../include/katsu_hip.h"
#include "split.hpp"
#include "splitconv.hpp"
#include "splitdw.hpp"
#include "splitgemm.hpp"

namespace katsu {
namespace {

constexpr int64_t kMaxElems = (int64_t)1 << 28;   // 1 GiB of floats
constexpr int64_t kMaxOffset = (int64_t)1 << 29;  // floats below 2^31 bytes
constexpr int kCUs = 256;
constexpr int kMaxLds = 160 * 1024;

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
// and costs a fixed part and a part per k.  Fitted to times measured before the
// operands were scaled (split3.hpp), which adds 2-8% to all of them: 256 x 128
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

// ---------------------------------------------------------------------------
// Convolutions.

template <int FM, int FN, int WPX, int WKG, int TG, int XU>
__global__ void __launch_bounds__(64 * WPX * WKG, 2) split_conv_kernel(const SplitConvArgs g) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    SplitConv<FM, FN, WPX, WKG, TG, XU>::run(g, lds, xcd_run(blockIdx.x, gridDim.x));
}

template <int FM, int FN, int WPX, int WKG, int TG, int XU>
int conv_launch(const SplitConvArgs &g, int64_t blocks, hipStream_t st) {
    using B = SplitConv<FM, FN, WPX, WKG, TG, XU>;
    constexpr auto kern = split_conv_kernel<FM, FN, WPX, WKG, TG, XU>;
    const int rc = lds_optin<kern>(kMaxLds);
    if (rc != KATSU_OK) return rc;
    kern<<<dim3((unsigned)blocks), dim3(B::kThreads), B::lds(g.slots), st>>>(g);
    return status_of(hipGetLastError());
}

constexpr int kMaxStrip = 64;

// Where a phase's tiles of BN pixels lie: strips of columns, pixels that tiles
// do not cross the ends of, tiles, and input pixels of a tile in LDS.
struct PhaseTiles {
    int NS, SW, PW;
    int64_t unit, utiles, tiles, slots;
};

PhaseTiles phase_tiles(const SplitPhase &p, int imgs, int st, int BN) {
    PhaseTiles t;
    t.NS = (int)cdiv(p.OW, kMaxStrip);
    t.SW = (int)cdiv(p.OW, t.NS);
    t.PW = (t.SW - 1) * st + p.Su;
    const int64_t strip = (int64_t)p.OH * t.SW, strips = (int64_t)imgs * t.NS;
    // Tiles end with their image's strip where that adds at most a tenth to
    // them: the rows between two images then take no LDS.
    const bool apart = cdiv(strip, BN) * BN * 10 <= strip * 11;
    t.unit = apart ? strip : strip * strips;
    t.utiles = cdiv(t.unit, BN);
    t.tiles = t.utiles * (apart ? strips : 1);
    const int64_t down = (t.SW - 1 + BN - 1) / t.SW;                 // output rows below the first
    const int64_t cross = apart ? 0 : (p.OH - 1 + down) / p.OH;      // image ends among them
    t.slots = (down * st + cross * std::max(0, p.Ru - st) + p.Ru) * t.PW;
    return t;
}

// A phase's fields as phase_tiles lays it out; its first tile is 0.
void phase_set(SplitPhase *p, const PhaseTiles &t, int imgs, int st) {
    p->NS = t.NS;
    p->SW = t.SW;
    p->PW = t.PW;
    p->Hs = (p->OH - 1) * st + p->Ru;
    p->taps = p->Ru * p->Su;
    p->unit = (int)t.unit;
    p->utiles = (int)t.utiles;
    p->npix = (int)((int64_t)imgs * t.NS * p->OH * t.SW);
    p->by_sw = split_div(p->SW);
    p->by_oh = split_div(p->OH);
    p->by_ns = split_div(p->NS);
    p->by_hs = split_div(p->Hs);
    p->by_pw = split_div(p->PW);
    p->by_su = split_div(p->Su);
    p->by_ut = split_div(p->utiles);
}

// The block shapes, and the time of a chunk of 16 channels at 9 taps, in ns:
// alone on a CU, and two blocks sharing it (measured on 3x3 layers: 512 ->
// 512 channels at 7 x 7, 256 -> 256 at 14 x 14 and 64 -> 64 at 56 x 56, batch
// 16-32).  The small tiles wait for their loads, the large ones approach the
// matrix rate, so a layer takes the largest tile that still fills the GPU.
//
// us: the whole launch in microseconds, for the choice between these kernels and
// the float32 ones: a fixed part, and per round of blocks one of the block, of a
// block whose stores are two pixels apart, of each chunk, of each chunk's tap, and
// of each chunk's input pixels per thread.  Of several phases the largest counts:
// an XCD holds a run of tiles, of one or two phases.  Fitted to 7600 runs over
// layers of 1 to 512 channels, filters of 1 to 9, both passes and strides: nine in
// ten take 0.87 to 1.2 of it.
struct ConvShape {
    int FM, FN, WPX, WKG, TG;
    double alone, shared;
    struct { double launch, block, apart, chunk, tap, slot; } us;
    constexpr int bm() const { return 32 * FM; }
    constexpr int bn() const { return 32 * FN * WPX; }
    constexpr int threads() const { return 64 * WPX * WKG; }
};
constexpr ConvShape kConvShapes[] = {
    {2, 2, 4, 1, 5, 9500, 14500, {4.4, 4.0, 2.8, 1.14, 0.78, 0}},
    {1, 2, 4, 1, 9, 5600, 7700, {3.3, 3.0, 0.6, 1.24, 0.41, 0}},
    {1, 1, 4, 2, 9, 3200, 4500, {2.2, 2.6, 1.0, 0.33, 0.227, 1.47}},
    {1, 1, 2, 4, 9, 2800, 3800, {0, 4.15, 1.4, 0.35, 0.176, 1.53}}};
constexpr int kNumConvShapes = 4;
constexpr int kMaxXU = 8;

template <int C>
using ConvOf = SplitConv<kConvShapes[C].FM, kConvShapes[C].FN, kConvShapes[C].WPX,
                         kConvShapes[C].WKG, kConvShapes[C].TG, 1>;
template <int... C>
constexpr int conv_lds_of(int c, int slots, std::integer_sequence<int, C...>) {
    int v = 0;
    ((c == C ? (void)(v = ConvOf<C>::lds(slots)) : (void)0), ...);
    return v;
}
int conv_lds(int c, int slots) {
    return conv_lds_of(c, slots, std::make_integer_sequence<int, kNumConvShapes>());
}

// The block shape of least estimated time, -1 if none takes the problem; *us:
// the launch in microseconds.
int conv_pick(const SplitConvArgs &g, double *us) {
    int best = -1;
    double t_best = 0;
    for (int c = 0; c < kNumConvShapes; ++c) {
        const ConvShape &s = kConvShapes[c];
        const int64_t tm = cdiv(g.CO, s.bm()), chunks = cdiv(g.CI, 16);
        int64_t blocks = 0, slots = 0;
        double taps = 0;
        int most_taps = 0;
        bool ok = true;
        for (int i = 0; i < g.nphases; ++i) {
            const SplitPhase &p = g.ph[i];
            const PhaseTiles t = phase_tiles(p, g.imgs, g.st, s.bn());
            const int64_t strips = (int64_t)g.imgs * t.NS;
            ok = ok && strips * p.OH * t.SW + s.bn() < (int64_t)1 << 31 &&
                 strips * ((p.OH - 1) * (int64_t)g.st + p.Ru) + 256 < (int64_t)1 << 31;
            slots = std::max(slots, t.slots);
            blocks += t.tiles * tm;
            // Below five taps a chunk is bound by its loads.
            taps += (double)t.tiles * tm * std::max(5, p.Ru * p.Su);
            most_taps = std::max(most_taps, p.Ru * p.Su);
        }
        if (!ok || 2 * slots > kMaxXU * s.threads() || blocks >= (int64_t)1 << 31) continue;
        const int lds = conv_lds(c, (int)slots);
        if (lds > kMaxLds) continue;
        // Registers of more than two blocks' waves fit for none of the shapes
        // at their usual sizes.
        const int64_t per_cu = lds <= kMaxLds / 2 ? 2 : 1;
        const int64_t full = blocks / (kCUs * per_cu), rest = blocks - full * kCUs * per_cu;
        const double round = per_cu == 2 ? s.shared : s.alone;
        const double rounds = (double)full * round + (rest > kCUs ? s.shared : rest ? s.alone : 0.);
        const double t = rounds * (double)chunks * taps / (double)blocks / 9.;
        if (best < 0 || t < t_best) {
            best = c;
            t_best = t;
            const double chunk = s.us.chunk + s.us.tap * most_taps +
                                 s.us.slot * (double)slots / s.threads();
            *us = s.us.launch + rounds / s.alone * (s.us.block + (g.osx > 1 ? s.us.apart : 0.) +
                                                    (double)chunks * chunk);
        }
    }
    return best;
}

template <int C>
int conv_go(SplitConvArgs &g, hipStream_t st) {
    constexpr ConvShape S = kConvShapes[C];
    g.slots = 0;
    g.tiles_m = (int)cdiv(g.CO, S.bm());
    int64_t tiles = 0;
    for (int i = 0; i < g.nphases; ++i) {
        SplitPhase &p = g.ph[i];
        const PhaseTiles t = phase_tiles(p, g.imgs, g.st, S.bn());
        phase_set(&p, t, g.imgs, g.st);
        p.tile0 = (int)tiles;
        g.slots = std::max(g.slots, (int)t.slots);
        tiles += t.tiles;
    }
    const int64_t blocks = tiles * g.tiles_m;
    // Input groups per thread.
    const int units = 2 * g.slots;
    if (units <= S.threads()) return conv_launch<S.FM, S.FN, S.WPX, S.WKG, S.TG, 1>(g, blocks, st);
    if (units <= 2 * S.threads())
        return conv_launch<S.FM, S.FN, S.WPX, S.WKG, S.TG, 2>(g, blocks, st);
    if (units <= 4 * S.threads())
        return conv_launch<S.FM, S.FN, S.WPX, S.WKG, S.TG, 4>(g, blocks, st);
    return conv_launch<S.FM, S.FN, S.WPX, S.WKG, S.TG, kMaxXU>(g, blocks, st);
}

// below: the time another kernel would take, in microseconds.
SplitRun conv_run(SplitConvArgs &g, double below, hipStream_t st, int *rc) {
    double us = 0;
    const int shape = conv_pick(g, &us);
    if (shape < 0) return SplitRun::kUnfit;
    // Both estimates are off by a tenth: with 3% to the other kernel's advantage
    // 1 layer in 100 is slower by more than a twentieth than with it, and 1 in 60
    // slower than here (without: 1 in 75 and 1 in 90).
    if (us * 1.03 >= below) return SplitRun::kSlower;
    switch (shape) {
        case 0: *rc = conv_go<0>(g, st); break;
        case 1: *rc = conv_go<1>(g, st); break;
        case 2: *rc = conv_go<2>(g, st); break;
        default: *rc = conv_go<3>(g, st); break;
    }
    return SplitRun::kLaunched;
}

bool layer_args(const SplitLayer &l, SplitConvArgs *g) {
    const int64_t nx = (int64_t)l.N * l.C * l.H * l.W, ny = (int64_t)l.N * l.K * l.OH * l.OW;
    const int64_t nw = (int64_t)l.K * l.C * l.R * l.S;
    if (nx >= kMaxElems || ny >= kMaxElems || nw >= kMaxElems || l.st > 2) return false;
    // The kernels' scalar offsets reach the end of a chunk of 16 channels, and in
    // the filter of the one after it: few channels of large planes (5 of 6000 x
    // 6000) would pass the 2^31 bytes that load1 allows.
    const int64_t cs = cdiv(l.C, 16) * 16, ks = cdiv(l.K, 16) * 16;
    if (cs * l.H * l.W >= kMaxOffset || ks * l.OH * l.OW >= kMaxOffset ||
        (ks + 16) * l.C * l.R * l.S >= kMaxOffset || (cs + 16) * l.R * l.S >= kMaxOffset)
        return false;
    *g = SplitConvArgs{};
    g->imgs = l.N;
    g->w_bytes = (uint32_t)(nw * 4);
    g->K = l.K;
    g->C = l.C;
    g->LH = l.H;
    g->LW = l.W;
    g->OH = l.OH;
    g->OW = l.OW;
    g->R = l.R;
    g->S = l.S;
    g->lst = l.st;
    g->lpad = l.pad;
    return true;
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

namespace {

bool fwd_args(const SplitLayer &l, SplitConvArgs *out) {
    SplitConvArgs &g = *out;
    if (!layer_args(l, &g)) return false;
    g.in_bytes = (uint32_t)((int64_t)l.N * l.C * l.H * l.W * 4);
    g.CI = l.C;
    g.CO = l.K;
    g.H = l.H;
    g.W = l.W;
    g.HW = l.H * l.W;
    g.st = l.st;
    g.in_img = l.C * g.HW;
    g.w_row = l.C * l.R * l.S;
    g.w_red = l.R * l.S;
    g.out_plane = l.OH * l.OW;
    g.out_img = (int64_t)l.K * g.out_plane;
    g.osy = l.OW;
    g.osx = 1;
    g.nphases = 1;
    SplitPhase &p = g.ph[0];
    p.OH = l.OH;
    p.OW = l.OW;
    p.pady = p.padx = l.pad;
    p.Ru = l.R;
    p.Su = l.S;
    p.tu = l.S;
    p.tv = 1;
    return true;
}

bool dx_args(const SplitLayer &l, SplitConvArgs *out) {
    SplitConvArgs &g = *out;
    if (!layer_args(l, &g)) return false;
    g.in_bytes = (uint32_t)((int64_t)l.N * l.K * l.OH * l.OW * 4);
    g.CI = l.K;
    g.CO = l.C;
    g.H = l.OH;
    g.W = l.OW;
    g.HW = l.OH * l.OW;
    g.st = 1;
    g.in_img = l.K * g.HW;
    g.w_row = l.R * l.S;
    g.w_red = l.C * l.R * l.S;
    g.out_plane = l.H * l.W;
    g.out_img = (int64_t)l.C * g.out_plane;
    g.osy = l.st * l.W;
    g.osx = l.st;
    g.dx = 1;
    for (int py = 0; py < l.st; ++py)
        for (int px = 0; px < l.st; ++px) {
            if (py >= l.H || px >= l.W) continue;
            // Input row py + st*a receives taps r = r0 + st*u from output row a + dy - u.
            const int r0 = (py + l.pad) % l.st, s0 = (px + l.pad) % l.st;
            if (r0 >= l.R || s0 >= l.S) return false;  // pixels no tap reaches
            SplitPhase &p = g.ph[g.nphases++];
            p.OH = (int)cdiv(l.H - py, l.st);
            p.OW = (int)cdiv(l.W - px, l.st);
            p.Ru = (int)cdiv(l.R - r0, l.st);
            p.Su = (int)cdiv(l.S - s0, l.st);
            p.pady = p.Ru - 1 - (py + l.pad - r0) / l.st;
            p.padx = p.Su - 1 - (px + l.pad - s0) / l.st;
            p.tu = -l.st * l.S;
            p.tv = -l.st;
            p.t0 = (r0 + l.st * (p.Ru - 1)) * l.S + s0 + l.st * (p.Su - 1);
            p.o0 = py * l.W + px;
        }
    return true;
}

}  // namespace

SplitRun split_conv_fwd(const float *x, const float *w, float *y, const SplitLayer &l,
                        double below, hipStream_t st, int *rc) {
    SplitConvArgs g;
    if (!fwd_args(l, &g)) return SplitRun::kUnfit;
    g.in = x;
    g.w = w;
    g.out = y;
    return conv_run(g, below, st, rc);
}

SplitRun split_conv_dx(const float *gy, const float *w, float *dx, const SplitLayer &l, float beta,
                       double below, hipStream_t st, int *rc) {
    SplitConvArgs g;
    if (!dx_args(l, &g)) return SplitRun::kUnfit;
    g.in = gy;
    g.w = w;
    g.out = dx;
    g.beta = beta;
    return conv_run(g, below, st, rc);
}

namespace {

template <int XU>
__global__ void __launch_bounds__(768, 3) split_dw_kernel(const SplitDwArgs g) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    SplitDw<XU>::run(g, lds, xcd_run(blockIdx.x, gridDim.x));
}

// Partial sums in the workspace: at most the 37.7 MB that the library's other
// plans need, which the static array of the allocation-free backward holds.
constexpr int64_t kMaxPartBytes = 37700000;

bool dw_args(const SplitLayer &l, SplitDwArgs *out) {
    using B = SplitDw<1>;
    SplitConvArgs f;
    if (!fwd_args(l, &f)) return false;
    SplitDwArgs &g = *out;
    g = SplitDwArgs{};
    g.x_bytes = f.in_bytes;
    g.g_bytes = (uint32_t)((int64_t)l.N * l.K * l.OH * l.OW * 4);
    g.C = l.C;
    g.K = l.K;
    g.H = l.H;
    g.W = l.W;
    g.HW = l.H * l.W;
    g.OHW = l.OH * l.OW;
    g.st = l.st;
    g.imgs = l.N;
    g.R = l.R;
    g.S = l.S;
    g.pad = l.pad;
    g.ph = f.ph[0];
    const PhaseTiles t = phase_tiles(g.ph, l.N, l.st, B::P);
    const int64_t npix = (int64_t)l.N * t.NS * l.OH * t.SW;
    if (npix + 2 * B::P >= (int64_t)1 << 31 ||
        (int64_t)l.N * t.NS * ((l.OH - 1) * (int64_t)l.st + l.R) + 256 >= (int64_t)1 << 31)
        return false;
    if (t.slots * (B::BC / 8) > 4 * B::kThreads || B::lds((int)t.slots) > kMaxLds) return false;
    phase_set(&g.ph, t, l.N, l.st);
    g.slots = (int)t.slots;
    g.tiles = (int)t.tiles;
    g.tiles_k = (int)cdiv(l.K, B::BK);
    g.tiles_c = (int)cdiv(l.C, B::BC);
    g.sets = (int)cdiv(g.ph.taps, 9);
    g.run_stride = ((int64_t)l.K * l.C * g.ph.taps + 3) / 4 * 4;
    // One block per CU, each with at least two tiles.
    const int64_t blocks = (int64_t)g.tiles_k * g.tiles_c * g.sets;
    int64_t runs = std::max<int64_t>(1, kCUs / blocks);
    runs = std::min(runs, std::max<int64_t>(1, g.tiles / 2));
    runs = std::min(runs, std::max<int64_t>(1, kMaxPartBytes / (g.run_stride * 4)));
    if (g.run_stride * 4 > kMaxPartBytes) return false;
    g.per_run = (int)cdiv(g.tiles, runs);
    g.runs = (int)cdiv(g.tiles, g.per_run);
    return blocks * g.runs < (int64_t)1 << 31;
}

template <int XU>
int dw_launch(const SplitDwArgs &g, hipStream_t st) {
    constexpr auto kern = split_dw_kernel<XU>;
    const int rc = lds_optin<kern>(kMaxLds);
    if (rc != KATSU_OK) return rc;
    const int64_t blocks = (int64_t)g.tiles_k * g.tiles_c * g.sets * g.runs;
    kern<<<dim3((unsigned)blocks), dim3(SplitDw<XU>::kThreads), SplitDw<XU>::lds(g.slots), st>>>(g);
    return status_of(hipGetLastError());
}

}  // namespace

size_t split_dw_bytes(const SplitLayer &l) {
    SplitDwArgs g;
    // Below 1.5 GFLOP of products the launch, the first loads and the partial sums'
    // reduction outweigh the matrix rate (one image of 64 -> 64 channels, 0.23
    // GFLOP: 31 us against 21; 128 -> 128 at 28 x 28, batch 8, 1.85 GFLOP: 38
    // against 45).  So do half-empty tiles of 64 x 32 channels and 9 taps (13 -> 15
    // channels 5x5: 266 against 205; 45 -> 83 channels 5x5: forward + backward 155
    // against 145; 128 -> 64 channels 1x1, padded: 155 against 62).  With
    // several sets of taps and few pixels the partial sums and their reduction
    // are most of the work (243 pixels, 427 -> 384 channels 5x5: 79 against 35; of
    // 170 such layers the middle one breaks even at 1000 pixels with 5x5 filters
    // and near 1700 with 7x7; with 3x3 ones all of 169 gain, down to 150 pixels).
    const int taps = l.R * l.S;
    const double flops = 2. * l.N * l.OH * l.OW * l.K * l.C * taps;
    const double fill = (double)l.K * l.C * taps /
                        ((double)cdiv(l.K, 64) * 64 * cdiv(l.C, 32) * 32 * cdiv(taps, 9) * 9);
    if (flops < 1.5e9 || fill < 0.5 || (taps > 9 && (int64_t)l.N * l.OH * l.OW < 1500)) return 0;
    return dw_args(l, &g) ? (size_t)(g.runs * g.run_stride) * sizeof(float) : 0;
}

int split_dw(const float *x, const float *gy, float *dw, const SplitLayer &l, float beta, float *ws,
             hipStream_t st) {
    SplitDwArgs g;
    if (!dw_args(l, &g)) return KATSU_E_INVALID;
    g.x = x;
    g.g = gy;
    g.part = ws;
    const int units = g.slots * (SplitDw<1>::BC / 8), th = SplitDw<1>::kThreads;
    const int rc = units <= th ? dw_launch<1>(g, st)
                   : units <= 2 * th ? dw_launch<2>(g, st) : dw_launch<4>(g, st);
    if (rc != KATSU_OK) return rc;
    const int64_t n = (int64_t)l.K * l.C * g.ph.taps;
    // Few runs: small blocks, whose threads then all have one to read.
    const dim3 blocks((unsigned)cdiv(n, 64));
    if (g.runs <= 32)
        split_dw_reduce<4><<<blocks, dim3(256), 0, st>>>(ws, dw, g.run_stride, g.runs, l.K * l.C,
                                                         g.ph.taps, beta);
    else
        split_dw_reduce<16><<<blocks, dim3(1024), 0, st>>>(ws, dw, g.run_stride, g.runs, l.K * l.C,
                                                           g.ph.taps, beta);
    return status_of(hipGetLastError());
}

}  // namespace katsu
