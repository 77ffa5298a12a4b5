// splitconv.hpp -- the convolution forward and data gradient on the bf16
// matrix cores (split3.hpp), any filter, stride 1 or 2 and padding.
//
// Both passes are one form: out[n][co][y][x] = sum over ci and taps (u, v) of
// w'[co][ci][u][v] * in[n][ci][y*st + u - pady][x*st + v - padx].  The data
// gradient of a stride-s layer is s*s of them (its phases), each at stride 1
// over G with the taps that reach that phase's pixels, as in igemm.hpp.
//
// A block computes 32 FM output channels over 32 FN WPX consecutive output
// pixels, counted through image rows and images.  Input channels come 16 at a
// time: the input rows that the pixels touch are loaded, split once and kept
// in LDS as [part][8 channels][pixel], so all taps read the same copy, each at
// its own offset (an im2col tile would be split again for every tap).  The
// filter comes TG taps at a time as [part][8 channels][tap][output channel].
// A matrix step is then 16 channels at one tap, and every fragment is one
// 16-byte LDS read per lane and part.
// WKG groups of waves share the tile and take every WKG-th tap; their sums
// meet in LDS, in order, at the end.
//
// What it runs at (batch 32, one MI355X, forward then dX; float32 kernels before):
// 64 -> 64 channels 3x3 at 56 x 56 61 (64) us forward, 256 -> 256 at 14 x 14 73
// (178) and 72 (314), 45 -> 83 5x5 at 37 x 51, batch 7, 39 (90) and 53 (216).
// What bounds it: waits, for the one chunk of loads in flight and at the barriers
// (a third of the waves' cycles); the matrix cores are 20-31% busy, the other
// vector instructions 19-34%, the LDS 15-27%, a quarter of it bank conflicts.
//
// Wide images are cut into strips of at most 64 columns, each treated as an
// image of its own, to bound the rows' length in LDS.
#pragma once

#include "exact.hpp"
#include "split3.hpp"
#include "splitgemm.hpp"

namespace katsu {

// Division of 0 <= n < 2^31 by a constant (Granlund & Montgomery, 1994), as
// igemm.hpp's FastDiv.
struct SplitDiv {
    uint32_t m, s;
    int d;
    __device__ __forceinline__ int div(int n) const {
        return (int)((__umulhi((uint32_t)n, m) + (uint32_t)n) >> s);
    }
};

inline SplitDiv split_div(uint32_t d) {
    SplitDiv f;
    const uint32_t s = d > 1 ? 32 - __builtin_clz(d - 1) : 0;
    f.d = (int)d;
    f.s = s;
    f.m = (uint32_t)(((1ull << 32) * ((1ull << s) - d)) / d + 1);
    return f;
}

// One phase: a grid of output pixels with its taps.
struct SplitPhase {
    int tile0;            // its first pixel tile
    int OH, OW, SW, NS;   // pixels; strip width and strips per row
    int Hs, PW;           // input rows per image, input columns per strip
    int pady, padx;
    int Ru, Su, taps;
    int t0, tu, tv;       // filter element of tap (u, v): t0 + u*tu + v*tv
    int o0;               // output element of pixel (0, 0) in its plane
    int npix;             // pixels of all images' strips, padding columns included
    int unit, utiles;     // pixels that tiles do not cross the ends of (an image's strip, or
                          // all), and tiles in them
    SplitDiv by_sw, by_oh, by_ns, by_hs, by_pw, by_su, by_ut;
};

struct SplitConvArgs {
    const float *in, *w;
    float *out;
    uint32_t in_bytes, w_bytes;
    int CI, CO, H, W, HW, st;
    int in_img, imgs;          // input floats per image; images
    int w_row, w_red;          // filter floats between output / input channels
    int out_plane, osy, osx;   // output floats between channels, rows, columns
    int64_t out_img;
    float beta;
    int tiles_m, nphases, slots;  // slots: input pixels of a tile in LDS, at most
    SplitPhase ph[4];
    // The layer, for values computed again (exact.hpp): dx says which pass.
    int dx, K, C, LH, LW, OH, OW, R, S, lst, lpad;
};

// One output value over the visited products, in their order.
__device__ __noinline__ float split_conv_exact(const float *in, const float *w, int dx, int K,
                                               int C, int LH, int LW, int OH, int OW, int R, int S,
                                               int st, int pad, int ch, int y, int x) {
    return dx ? exact_dx_inl(in, w, K, C, OH, OW, R, S, st, pad, ch, y, x)
              : exact_fwd_inl(in, w, C, LH, LW, R, S, st, pad, ch, y, x);
}

template <int FM, int FN, int WPX, int WKG, int TG, int XU>
struct SplitConv {
    static constexpr int kThreads = 64 * WPX * WKG;
    static constexpr int BM = 32 * FM, BN = 32 * FN * WPX;
    static constexpr int kTap = BM * 16 + 16;          // bytes of one tap's 8-channel rows
    static constexpr int kWPlane = TG * kTap;
    static constexpr int kWBytes = 6 * kWPlane;
    static constexpr int kUnits = 2 * BM * TG;         // 8-channel groups of a filter stage
    static constexpr int WU = (kUnits + kThreads - 1) / kThreads;
    static constexpr int kRun = 9;  // matrix steps of 16 products summed before the total takes them
    static constexpr int kSum = WPX * WKG * FM * FN * 4096;  // the waves' sums

    static constexpr int plane(int slots) { return slots * 16 + 32; }
    static constexpr int lds(int slots) {
        const int a = kWBytes + 6 * plane(slots);
        return a > kSum ? a : kSum;
    }

    __device__ static void run(const SplitConvArgs &g, char *lds, int t) {
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int wpx = wave % WPX, wkg = wave / WPX;
        int phase = 0;
        const int tm = t % g.tiles_m, tn_all = t / g.tiles_m;
        while (phase + 1 < g.nphases && tn_all >= g.ph[phase + 1].tile0) ++phase;
        const SplitPhase &P = g.ph[phase];
        const int co0 = tm * BM, ti = tn_all - P.tile0, un = P.by_ut.div(ti);
        const int q0 = un * P.unit + (ti - un * P.utiles) * BN, qend = (un + 1) * P.unit;
        const int st = g.st;

        // First input row, counted over all images' strips.
        const int g0 = P.by_sw.div(q0);
        const int im0 = P.by_oh.div(g0);
        const int Y0 = im0 * P.Hs + (g0 - im0 * P.OH) * st;

        const __amdgpu_buffer_rsrc_t rin = split_rsrc(g.in, g.in_bytes);
        const __amdgpu_buffer_rsrc_t rw = split_rsrc(g.w, g.w_bytes);
        const int xplane = plane(g.slots);
        char *lw = lds, *lx = lds + kWBytes;

        // This thread's input groups: byte offset of channel 0 (or out of
        // range: padding), LDS place.
        int xoff[XU], xdst[XU];
        const int slots = g.slots;
#pragma unroll
        for (int e = 0; e < XU; ++e) {
            const int u = tid + e * kThreads;
            const int cg = u >= slots ? 1 : 0, slot = u - cg * slots;
            xdst[e] = -1;
            xoff[e] = kSplitOOB;
            if (u < 2 * slots) {
                const int row = P.by_pw.div(slot), col = slot - row * P.PW;
                const int Y = Y0 + row, im = P.by_hs.div(Y);
                const int n = P.by_ns.div(im);
                const int iy = Y - im * P.Hs - P.pady;
                const int ix = (im - n * P.NS) * P.SW * st + col - P.padx;
                xdst[e] = cg * xplane + slot * 16;
                if (n < g.imgs && (unsigned)iy < (unsigned)g.H && (unsigned)ix < (unsigned)g.W &&
                    cg * 8 < g.CI)
                    xoff[e] = (n * g.in_img + cg * 8 * g.HW + iy * g.W + ix) * 4;
            }
        }
        // Its filter groups: tap fastest, so that lanes read runs of memory.
        int woff[WU], wdst[WU], wtap[WU], wlast[WU];
#pragma unroll
        for (int e = 0; e < WU; ++e) {
            const int u = tid + e * kThreads;
            const int tl = u % TG, row = u / TG % BM, cg = u / (TG * BM);
            wtap[e] = u < kUnits && co0 + row < g.CO ? tl : 1 << 16;
            wlast[e] = g.CI - cg * 8;
            woff[e] = (co0 + row) * g.w_row + cg * 8 * g.w_red;
            wdst[e] = u < kUnits ? cg * kWPlane + tl * kTap + row * 16 : -1;
        }
        // This lane's pixels: LDS offset of their tap (0, 0).
        int pix[FN];
#pragma unroll
        for (int b = 0; b < FN; ++b) {
            const int q = min(q0 + (wpx * FN + b) * 32 + (lane & 31), qend - 1);
            const int gr = P.by_sw.div(q), im = P.by_oh.div(gr);
            const int Y = im * P.Hs + (gr - im * P.OH) * st;
            pix[b] = ((Y - Y0) * P.PW + (q - gr * P.SW) * st) * 16 + (lane >> 5) * xplane;
        }
        const int arow = (lane >> 5) * kWPlane + (lane & 31) * 16;

        floatx16 tot[FM][FN], acc[FM][FN];
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int b = 0; b < FN; ++b) tot[a][b] = acc[a][b] = floatx16{};

        float xr[XU][8], wr[WU][8];
        // Input channels past the last read the next image, or zeros past the
        // tensor (load1's range check): their filter values are zeros, and a
        // product that is then not finite is computed again like any other.
        // (Lanes' offsets selected in the last chunk instead: forward + backward
        // of 64 -> 64 channels 3x3 at 56 x 56, batch 32, 189 -> 221 us.)
        auto load_x = [&](int so) {
#pragma unroll
            for (int e = 0; e < XU; ++e)
#pragma unroll
                for (int i = 0; i < 8; ++i) xr[e][i] = load1(rin, xoff[e], so + i * g.HW * 4);
        };
        const int su = P.Su, taps = P.taps, pw = P.PW, wt0 = P.t0, wtu = P.tu, wtv = P.tv;
        const SplitDiv by_su = P.by_su;
        auto load_w = [&](int c0, int g0t) {
#pragma unroll
            for (int e = 0; e < WU; ++e) {
                const int tg = g0t + wtap[e], u = by_su.div(tg);
                const int o = tg < taps ? (woff[e] + wt0 + u * wtu + (tg - u * su) * wtv) * 4
                                        : kSplitOOB;
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    wr[e][i] = load1(rw, c0 + i < wlast[e] ? o : kSplitOOB, (c0 + i) * g.w_red * 4);
            }
        };

        const int chunks = (g.CI + 15) / 16, groups = (taps + TG - 1) / TG;
        // The total takes the sums after whole chunks, about every kSplitFlush
        // products, and between groups of taps before a wave passes kRun steps.
        const int flush_every = max(1, kSplitFlush / (16 * taps));
        auto flush = [&] {
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) {
                    tot[a][b] += acc[a][b];
                    acc[a][b] = floatx16{};
                }
        };
        auto steps = [](int n) { return (n + WKG - 1) / WKG; };
        load_x(0);
        load_w(0, 0);
        int flush_in = flush_every, run = 0;
        for (int c = 0; c < chunks; ++c) {
#pragma unroll
            for (int e = 0; e < XU; ++e) {
                uintx4 s[3];
                split3(xr[e], s);
                if (xdst[e] >= 0)
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        *reinterpret_cast<uintx4 *>(lx + xdst[e] + q * 2 * xplane) = s[q];
            }
            for (int gt = 0; gt < groups; ++gt) {
#pragma unroll
                for (int e = 0; e < WU; ++e) {
                    uintx4 s[3];
                    split3(wr[e], s);
                    if (wdst[e] >= 0)
#pragma unroll
                        for (int q = 0; q < 3; ++q)
                            *reinterpret_cast<uintx4 *>(lw + wdst[e] + q * 2 * kWPlane) = s[q];
                }
                __syncthreads();
                const bool last = gt + 1 == groups;
                load_w((last ? c + 1 : c) * 16, last ? 0 : (gt + 1) * TG);
                // After the last chunk: out of range, which reads no memory.
                if (gt == 0) load_x(c + 1 < chunks ? (c + 1) * 16 * g.HW * 4 : kSplitEnd);
                __builtin_amdgcn_sched_barrier(kSchedNoVmem);
                const int t0 = gt * TG, nt = min(TG, taps - t0);
                for (int tl = wkg; tl < nt; tl += WKG) {
                    const int u = by_su.div(t0 + tl), v = t0 + tl - u * su;
                    const int bo = (u * pw + v) * 16, ao = tl * kTap + arow;
                    uintx4 af[FM][3], bf[FN][3];
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
#pragma unroll
                        for (int a = 0; a < FM; ++a)
                            af[a][q] = *reinterpret_cast<const uintx4 *>(lw + ao + q * 2 * kWPlane +
                                                                         a * 512);
#pragma unroll
                        for (int b = 0; b < FN; ++b)
                            bf[b][q] = *reinterpret_cast<const uintx4 *>(lx + pix[b] + bo +
                                                                         q * 2 * xplane);
                    }
#pragma unroll
                    for (int q = 0; q < 6; ++q)
#pragma unroll
                        for (int a = 0; a < FM; ++a)
#pragma unroll
                            for (int b = 0; b < FN; ++b)
                                acc[a][b] = mfma32(af[a][kSplitA[q]], bf[b][kSplitB[q]], acc[a][b]);
                }
                __syncthreads();
                if (!last) {
                    run += steps(nt);
                    if (run + steps(min(TG, taps - t0 - TG)) > kRun) {
                        run = 0;
                        flush();
                    }
                }
            }
            if (--flush_in == 0 || c + 1 == chunks) {
                flush_in = flush_every;
                flush();
            }
            run = 0;
        }

        // The wave groups' sums, added in order by the first group.
        if constexpr (WKG > 1) {
            floatx16 *s = reinterpret_cast<floatx16 *>(lds);
            if (wkg > 0)
#pragma unroll
                for (int a = 0; a < FM; ++a)
#pragma unroll
                    for (int b = 0; b < FN; ++b)
                        s[((wkg * WPX + wpx) * FM * FN + a * FN + b) * 64 + lane] = tot[a][b];
            __syncthreads();
            if (wkg > 0) return;
#pragma unroll
            for (int k = 1; k < WKG; ++k)
#pragma unroll
                for (int a = 0; a < FM; ++a)
#pragma unroll
                    for (int b = 0; b < FN; ++b)
                        tot[a][b] += s[((k * WPX + wpx) * FM * FN + a * FN + b) * 64 + lane];
        }

        bool bad = false;
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int b = 0; b < FN; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    bad |= !__builtin_isfinite(tot[a][b][v]);
                    tot[a][b][v] *= kSplitUnscale;
                }
        const bool redo = __any(bad);
        // The wave's own part of the LDS, which nothing reads any more: the
        // rare recomputation then is a loop over values in memory, outside the
        // straight code of the stores.
        floatx16 *own = reinterpret_cast<floatx16 *>(lds) + wave * FM * FN * 64 + lane;
        if (redo)
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) own[(a * FN + b) * 64] = tot[a][b];
#pragma unroll
        for (int b = 0; b < FN; ++b) {
            const int q = q0 + (wpx * FN + b) * 32 + (lane & 31);
            const int gr = P.by_sw.div(q), im = P.by_oh.div(gr), n = P.by_ns.div(im);
            const int y = gr - im * P.OH, x = (im - n * P.NS) * P.SW + q - gr * P.SW;
            if (q >= qend || x >= P.OW) continue;
            const int o = P.o0 + y * g.osy + x * g.osx;
            const int ch0 = co0 + 4 * (lane >> 5);
            float *dst = g.out + (int64_t)n * g.out_img + o + (int64_t)ch0 * g.out_plane;
            if (redo) {
                for (int i = 0; i < FM * 16; ++i) {
                    const int cl = i / 4 * 8 + i % 4;
                    if (ch0 + cl >= g.CO) continue;
                    float val = reinterpret_cast<const float *>(own + (i / 16 * FN + b) * 64)[i % 16];
                    if (!__builtin_isfinite(val))
                        val = split_conv_exact(
                            g.in + (int64_t)n * g.in_img, g.w, g.dx, g.K, g.C, g.LH, g.LW, g.OH,
                            g.OW, g.R, g.S, g.lst, g.lpad, ch0 + cl, g.dx ? o / g.LW : y,
                            g.dx ? o % g.LW : x);
                    float *p = dst + (int64_t)cl * g.out_plane;
                    *p = g.beta == 0.f ? val : g.beta * *p + val;
                }
            } else if (co0 + BM <= g.CO && g.beta == 0.f) {
#pragma unroll
                for (int i = 0; i < FM * 16; ++i)
                    dst[(int64_t)(i / 4 * 8 + i % 4) * g.out_plane] = tot[i / 16][b][i % 16];
            } else {
#pragma unroll
                for (int i = 0; i < FM * 16; ++i) {
                    const int cl = i / 4 * 8 + i % 4;
                    if (ch0 + cl >= g.CO) continue;
                    float *p = dst + (int64_t)cl * g.out_plane;
                    *p = g.beta == 0.f ? tot[i / 16][b][i % 16] : g.beta * *p + tot[i / 16][b][i % 16];
                }
            }
        }
    }
};

}  // namespace katsu
