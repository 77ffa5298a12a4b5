// splitdw.hpp -- the convolution's filter gradient on the bf16 matrix cores
// (split3.hpp), any filter, stride 1 or 2 and padding.
//
// dw[k][c][r][s] = sum over output pixels of gy[pixel][k] * x[pixel*st + tap][c].
// The reduction runs over pixels, which the matrix instruction wants
// contiguous per lane, while memory order and the taps' shifts want them as
// whole pixels.  Both operands are therefore kept in LDS as in splitconv.hpp,
// [part][8 channels][pixel], split once for all taps, and read with the
// transposing LDS load: four lanes name a pixel's 16 channels, and each lane
// gets one channel of four pixels.  A tap is then an offset added to the
// pixels' places, whatever the stride.
//
// A block: 64 output by 32 input channels, up to 9 taps, and a run of pixel
// tiles of 128.  Its 12 waves are 2 (halves of the output channels) x 3
// (groups of 3 taps) x 2 (every other 16 pixels); the last two meet in LDS at
// the end.  The partial sums of all runs go to the workspace as
// [run][tap][output channel][input channel], where a wave's stores are whole
// 128-byte lines, and split_dw_reduce adds them in order.
//
// Measured (one MI355X, the reduction included; float32 kernels before): 256 -> 256
// channels 3x3 at 14 x 14, batch 32, 68 us (139); 512 -> 512 at 7 x 7, batch 16, 58
// (111); 96 -> 96 5x5 at 56 x 56, batch 16, 297 (529).  Of the 78 us that 64 -> 64
// at 56 x 56 took, 32 are matrix instructions and their reads, 14 waits for
// loads, 6 the split, and the rest start, partial sums and their reduction.
#pragma once

#include "splitconv.hpp"

namespace katsu {

typedef short shortx4 __attribute__((ext_vector_type(4)));

struct SplitDwArgs {
    const float *x, *g;
    float *part;
    uint32_t x_bytes, g_bytes;
    int C, K, H, W, HW, OHW, st, imgs;
    int R, S, pad;
    int tiles_k, tiles_c, sets;   // blocks of 64 and 32 channels, sets of 9 taps
    int tiles, runs, per_run;     // pixel tiles, split into runs
    int slots;
    int64_t run_stride;           // floats between runs
    SplitPhase ph;                // the layer's output pixels and taps
};

// One dw value over the pixels [q0, q1), counted through the strips as the
// tiles are, over the visited products only.
__device__ __noinline__ float split_dw_exact(const float *x, const float *g, int C, int K, int H,
                                             int W, int OH, int OW, int SW, int NS, int st, int pad,
                                             int k, int c, int r, int s, int q0, int q1) {
#pragma clang fp contract(off)
    float acc = 0.f;
    int xs = q0 % SW, gr = q0 / SW;
    int y = gr % OH, im = gr / OH;
    for (int q = q0; q < q1; ++q) {
        const int n = im / NS, ox = (im - n * NS) * SW + xs;
        const int iy = y * st + r - pad, ix = ox * st + s - pad;
        if (ox < OW && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W)
            acc = acc + g[(((int64_t)n * K + k) * OH + y) * OW + ox] *
                            x[(((int64_t)n * C + c) * H + iy) * W + ix];
        if (++xs == SW) {
            xs = 0;
            if (++y == OH) {
                y = 0;
                ++im;
            }
        }
    }
    return acc;
}

template <int XU>
struct SplitDw {
    static constexpr int BK = 64, BC = 32, P = 128, TPW = 3;
    static constexpr int kThreads = 768;
    static constexpr int GU = 2;                       // P * BK/8 groups over 768 threads
    // Planes of 8 channels 64 bytes apart (mod 256): the four that a transposing
    // load reads, 64 bytes of each, then fall on different banks.
    static constexpr int kGPlane = P * 16 + 64;
    static constexpr int kGPart = BK / 8 * kGPlane;
    static constexpr int kGBytes = 3 * kGPart;
    static constexpr int kTable = P * 4;
    static constexpr int kSum = 6 * TPW * 4096;

    static constexpr int xplane(int slots) { return (slots * 16 + 255) / 256 * 256 + 64; }
    static constexpr int lds(int slots) {
        const int a = kTable + kGBytes + 3 * BC / 8 * xplane(slots);
        return a > 2 * kSum ? a : 2 * kSum;  // both pixel halves' sums
    }

    // Four pixels of one channel: lane l of 16 names pixel l/4's channels
    // 4 (l%4).. at `p` and gets channel l.
    static __device__ __forceinline__ uint64_t read_tr(const char *p) {
        typedef __attribute__((address_space(3))) shortx4 *lds_ptr;
        return __builtin_bit_cast(uint64_t,
                                  __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p)));
    }

    __device__ static void run(const SplitDwArgs &g, char *lds, int t) {
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int wk = wave % 2, wt = wave / 2 % 3, wp = wave / 6;
        const SplitPhase &P0 = g.ph;
        // Blocks of one run are neighbours: they read the same pixels.
        const int tk = t % g.tiles_k, tc = t / g.tiles_k % g.tiles_c;
        const int set = t / (g.tiles_k * g.tiles_c) % g.sets;
        const int rn = t / (g.tiles_k * g.tiles_c * g.sets);
        const int k0 = tk * BK, c0 = tc * BC;
        const int tile0 = rn * g.per_run, tile1 = min(tile0 + g.per_run, g.tiles);

        const __amdgpu_buffer_rsrc_t rx = split_rsrc(g.x, g.x_bytes);
        const __amdgpu_buffer_rsrc_t rg = split_rsrc(g.g, g.g_bytes);
        const int xp = xplane(g.slots);
        int *table = reinterpret_cast<int *>(lds);
        char *lg = lds + kTable, *lx = lg + kGBytes;

        // This thread's groups of 8 channels.  G: one pixel (768 is a multiple
        // of 128), two groups; x: pixels of the tile's rows.
        const int gp = tid % P, gk = tid / P;                 // 0..5, then + 6
        int xrow[XU], xcol[XU], xcg[XU], xdst[XU];
#pragma unroll
        for (int e = 0; e < XU; ++e) {
            const int u = tid + e * kThreads;
            const int cg = u / g.slots, slot = u - cg * g.slots;
            xrow[e] = P0.by_pw.div(slot);
            xcol[e] = slot - xrow[e] * P0.PW - P0.padx;
            xcg[e] = cg < BC / 8 && c0 + cg * 8 < g.C ? (c0 + cg * 8) * g.HW : -1;
            xdst[e] = cg < BC / 8 ? cg * xp + slot * 16 : -1;
        }

        float gr_[GU][8], xr[XU][8];
        int slot_next = 0;  // LDS place of pixel gp of the tile being loaded
        auto load = [&](int tile) {
            const int un = P0.by_ut.div(tile);
            const int q0 = un * P0.unit + (tile - un * P0.utiles) * P;
            const int qend = tile < tile1 ? (un + 1) * P0.unit : 0;
            const int g0 = P0.by_sw.div(q0), im0 = P0.by_oh.div(g0);
            const int Y0 = im0 * P0.Hs + (g0 - im0 * P0.OH) * g.st;
            // G at this thread's pixel.
            const int q = q0 + gp, gr = P0.by_sw.div(q), im = P0.by_oh.div(gr), n = P0.by_ns.div(im);
            const int y = gr - im * P0.OH, xs = q - gr * P0.SW, ox = (im - n * P0.NS) * P0.SW + xs;
            const bool in = q < qend && ox < P0.OW;
            const int Y = im * P0.Hs + y * g.st;
            slot_next = in ? ((Y - Y0) * P0.PW + xs * g.st) * 16 : 0;
            // Groups that begin past the last channel read zeros; the others' end
            // reads the next image's first channels, whose sums are not stored.
            const int go = n * g.K * g.OHW + y * P0.OW + ox;
#pragma unroll
            for (int e = 0; e < GU; ++e) {
                const int k = k0 + (gk + e * 6) * 8;
                const int o = in && k < g.K ? (go + k * g.OHW) * 4 : kSplitOOB;
#pragma unroll
                for (int i = 0; i < 8; ++i) gr_[e][i] = load1(rg, o, i * g.OHW * 4);
            }
#pragma unroll
            for (int e = 0; e < XU; ++e) {
                const int Yx = Y0 + xrow[e], imx = P0.by_hs.div(Yx), nx = P0.by_ns.div(imx);
                const int iy = Yx - imx * P0.Hs - P0.pady;
                const int ix = (imx - nx * P0.NS) * P0.SW * g.st + xcol[e];
                const bool ok = tile < tile1 && nx < g.imgs && (unsigned)iy < (unsigned)g.H &&
                                (unsigned)ix < (unsigned)g.W && xcg[e] >= 0;
                const int o = ok ? (nx * g.C * g.HW + xcg[e] + iy * g.W + ix) * 4 : kSplitOOB;
#pragma unroll
                for (int i = 0; i < 8; ++i) xr[e][i] = load1(rx, o, i * g.HW * 4);
            }
        };

        // Fragment reads: this lane's pixel in 16 (and 4 on), its channels.
        const int m = lane & 15, half = lane >> 5, hi = (lane >> 4) & 1;
        const int pk = half * 8 + m / 4;
        const int chan = (hi * 2 + (m >> 1 & 1)) , sub = (m & 1) * 8;
        const int gbase = (wk * 4 + chan) * kGPlane + sub + pk * 16;
        const int xbase = chan * xp + sub;
        int toff[TPW];
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            const int tp = min(set * 9 + wt * TPW + i, P0.taps - 1), u = P0.by_su.div(tp);
            toff[i] = (u * P0.PW + tp - u * P0.Su) * 16;
        }
        const int my_taps = min(TPW, P0.taps - set * 9 - wt * TPW);

        floatx16 tot[TPW], acc[TPW];
#pragma unroll
        for (int i = 0; i < TPW; ++i) tot[i] = acc[i] = floatx16{};

        load(tile0);
        for (int tile = tile0; tile < tile1; ++tile) {
            if (tid < P) table[tid] = slot_next;
#pragma unroll
            for (int e = 0; e < GU; ++e) {
                uintx4 s[3];
                split3(gr_[e], s);
                if (gk + e * 6 < BK / 8)
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        *reinterpret_cast<uintx4 *>(lg + (gk + e * 6) * kGPlane + gp * 16 +
                                                    q * kGPart) = s[q];
            }
#pragma unroll
            for (int e = 0; e < XU; ++e) {
                uintx4 s[3];
                split3(xr[e], s);
                if (xdst[e] >= 0)
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        *reinterpret_cast<uintx4 *>(lx + xdst[e] + q * (BC / 8) * xp) = s[q];
            }
            __syncthreads();
            load(tile + 1);
            __builtin_amdgcn_sched_barrier(kSchedNoVmem);
            for (int ks = wp; ks < P / 16; ks += 2) {
                if (my_taps <= 0) break;
                uintx4 af[3];
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    const char *p = lg + gbase + ks * 256 + q * kGPart;
                    const uint64_t a = read_tr(p), b = read_tr(p + 64);
                    af[q] = uintx4{(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)};
                }
                const int s0 = table[ks * 16 + pk], s1 = table[ks * 16 + pk + 4];
#pragma unroll
                for (int i = 0; i < TPW; ++i) {
                    uintx4 bf[3];
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        const char *p = lx + xbase + toff[i] + q * (BC / 8) * xp;
                        const uint64_t a = read_tr(p + s0), b = read_tr(p + s1);
                        bf[q] =
                            uintx4{(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)};
                    }
#pragma unroll
                    for (int q = 0; q < 6; ++q)
                        acc[i] = mfma32(af[kSplitA[q]], bf[kSplitB[q]], acc[i]);
                }
            }
            // A tile is 64 pixels per wave: short sums, added in float32.
#pragma unroll
            for (int i = 0; i < TPW; ++i) {
                tot[i] += acc[i];
                acc[i] = floatx16{};
            }
            __syncthreads();
        }

        // The two pixel halves' sums.
        floatx16 *own = reinterpret_cast<floatx16 *>(lds) + wave * TPW * 64 + lane;
        if (wp == 1)
#pragma unroll
            for (int i = 0; i < TPW; ++i) own[i * 64] = tot[i];
        __syncthreads();
        if (wp == 1) return;
#pragma unroll
        for (int i = 0; i < TPW; ++i) tot[i] += own[(6 * TPW + i) * 64];

        const int c = c0 + (lane & 31);
        float *dst = g.part + rn * g.run_stride + c;
        bool bad = false;
#pragma unroll
        for (int i = 0; i < TPW; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                bad |= !__builtin_isfinite(tot[i][v]);
                tot[i][v] *= kSplitUnscale;
            }
        if (__any(bad)) {
            const int un0 = P0.by_ut.div(tile0), un1 = P0.by_ut.div(tile1);
            const int q0 = un0 * P0.unit + (tile0 - un0 * P0.utiles) * P;
            const int q1 = min(un1 * P0.unit + (tile1 - un1 * P0.utiles) * P, P0.npix);
#pragma unroll
            for (int i = 0; i < TPW; ++i) own[i * 64] = tot[i];
            for (int e = 0; e < TPW * 16; ++e) {
                const int i = e / 16, v = e % 16, tp = set * 9 + wt * TPW + i;
                const int k = k0 + wk * 32 + 8 * (v / 4) + 4 * half + v % 4;
                if (i >= my_taps || k >= g.K || c >= g.C) continue;
                float val = reinterpret_cast<const float *>(own + i * 64)[v];
                if (!__builtin_isfinite(val))
                    val = split_dw_exact(g.x, g.g, g.C, g.K, g.H, g.W, P0.OH, P0.OW, P0.SW, P0.NS,
                                         g.st, g.pad, k, c, tp / g.S, tp % g.S, q0, q1);
                dst[((int64_t)tp * g.K + k) * g.C] = val;
            }
            return;
        }
        if (c >= g.C) return;
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            if (i >= my_taps) break;
            const int tp = set * 9 + wt * TPW + i;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int k = k0 + wk * 32 + 8 * (v / 4) + 4 * half + v % 4;
                if (k < g.K) dst[((int64_t)tp * g.K + k) * g.C] = tot[i][v];
            }
        }
    }
};

// dw[k][c][tap] = beta*dw + the sum of the runs' [tap][k][c], in a fixed order:
// GROUPS groups of 64 threads take every GROUPS-th run, their sums are added in
// order.
template <int GROUPS>
__global__ void __launch_bounds__(64 * GROUPS) split_dw_reduce(const float *part, float *dw, int64_t stride,
                                                        int runs, int KC, int taps, float beta) {
    __shared__ float s[GROUPS][64];
    const int l = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int64_t e = (int64_t)blockIdx.x * 64 + l, n = (int64_t)KC * taps;
    float v = 0.f;
    if (e < n) {
        const float *p = part + e;
#pragma unroll 8
        for (int r = grp; r < runs; r += GROUPS) v += p[r * stride];
    }
    s[grp][l] = v;
    __syncthreads();
    if (grp || e >= n) return;
#pragma unroll
    for (int i = 1; i < GROUPS; ++i) v += s[i][l];
    const int tap = (int)(e / KC), kc = (int)(e - (int64_t)tap * KC);
    float *o = dw + (int64_t)kc * taps + tap;
    *o = beta == 0.f ? v : beta * *o + v;
}

}  // namespace katsu
