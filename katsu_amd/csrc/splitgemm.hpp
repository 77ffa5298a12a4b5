// splitgemm.hpp -- the float32 GEMM on the bf16 matrix cores (split3.hpp).
//
// C[M,N] = beta*C + op(A) op(B), any sizes, any alignment of float pointers.
//
// A block computes a BM x BN tile, each wave WM x WN of it in fragments of
// 32 x 32.  A stage is 32 deep in k: the threads load their share of both
// operands as floats (one stage ahead, in registers), split it and write it
// to LDS as [part][k/8][row][8 bf16], so a fragment is one 16-byte read per
// lane and part, and 16 lanes read 256 contiguous bytes.  The k/8 planes are
// 32 bytes (mod 128) apart beyond a whole number of rows: the writers of a
// k-contiguous operand (four neighbouring lanes hold the four k/8 of one row)
// then fall on different banks.
#pragma once

#include "split3.hpp"

namespace katsu {

struct SplitGemmArgs {
    const float *a, *b;
    float *c;
    int M, N, K;
    int lda, ldb, ldc;
    uint32_t a_bytes, b_bytes;    // each below 1 GiB: operands are read at 32-bit buffer offsets
    float beta;
    int tiles_m, tiles_n, group;  // group: tile rows walked together
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t split_rsrc(const float *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), (short)0, (int)bytes,
                                             0x00020000);
}
// Floats at byte offset off (per lane) + so (the wave's): one, or eight in a
// row.  A buffer load needs 4-byte alignment only, whatever its width.  The
// range check counts both parts (measured with 1024 bytes described and off
// 0..504: so = 768 returns the first 256 bytes' lanes and zeros, so = 24000
// zeros), so what lies past the operand's end reads zero.  off + so as unsigned
// numbers stay below 2^32 in every call: operands end below 2^30; off lies in
// the operand or is kSplitOOB; so lies in it, at most 31 k (31 channels) past it
// or 7 channels past kSplitEnd, and below 2^31.
__device__ __forceinline__ float load1(__amdgpu_buffer_rsrc_t r, int off, int so) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, so, 0));
}
__device__ __forceinline__ void load8(__amdgpu_buffer_rsrc_t r, int off, int so, float (&v)[8]) {
    const floatx4 u = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, off, so, 0));
    const floatx4 w =
        __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 16, so, 0));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[i] = u[i];
        v[4 + i] = w[i];
    }
}

// A scheduling fence for loads only: the compiler would sink them to their use.
constexpr int kSchedNoVmem = 0x38f;
// A byte offset beyond any operand: such a load returns zero.
constexpr int kSplitOOB = (int)0x80000000;
constexpr int kSplitEnd = 1 << 30;  // the end of the largest operand
constexpr int kSplitFlush = 128;  // k summed on the matrix cores before the total takes them

// One operand's tile of BI rows by BK k.  KC: the operand is contiguous
// along k in memory, else along its rows.
template <int BI, int BK, int THREADS, bool KC>
struct SplitTile {
    static constexpr int kPlane = BI * 16 + 32;            // bytes of one k/8
    static constexpr int G = BK / 8;
    static constexpr int kPart = G * kPlane;
    static constexpr int kBytes = 3 * kPart;
    static constexpr int E = BI * G / THREADS;             // 8-float groups per thread
    static_assert(E >= 1 && BI * G % THREADS == 0, "tile/threads mismatch");

    __amdgpu_buffer_rsrc_t rs;
    int off[KC ? E : 1];  // byte offset of each group's first k (KC), else of the thread's
    int dst[E];           // LDS byte offset of each group
    int kg0;              // first k of this thread's group 0
    int ld4;              // bytes between rows (KC) or between k

    __device__ __forceinline__ void init(const float *base, uint32_t bytes, int ld, int i0, int I,
                                         int tid) {
        rs = split_rsrc(base, bytes);
        ld4 = ld * 4;
        if constexpr (KC) {
            kg0 = tid % G * 8;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int row = tid / G + e * (THREADS / G);
                off[e] = min(i0 + row, I - 1) * ld4 + kg0 * 4;
                dst[e] = tid % G * kPlane + row * 16;
            }
        } else {
            // Lanes along the rows; with fewer threads than BI BK/8 a
            // thread takes several k/8 of one row.
            const int row = tid % BI, g = tid / BI * E;
            kg0 = g * 8;
            off[0] = kg0 * ld4 + min(i0 + row, I - 1) * 4;
#pragma unroll
            for (int e = 0; e < E; ++e) dst[e] = (g + e) * kPlane + row * 16;
        }
    }
    // The stage at k0; left: its k that exist, at least BK with FULL.  A k
    // past the end is read at an offset out of the buffer's range, as zero.
    template <bool FULL>
    __device__ __forceinline__ void load(float (&r)[E][8], int k0, int left) const {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            if constexpr (KC && FULL) {
                load8(rs, off[e], k0 * 4, r[e]);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int k = KC ? i : e * 8 + i;
                    const bool in = FULL || kg0 + k < left;
                    r[e][i] = KC ? load1(rs, in ? off[e] + 4 * i : kSplitOOB, k0 * 4)
                                 : load1(rs, in ? off[0] : kSplitOOB, (k0 + k) * ld4);
                }
            }
        }
    }
    __device__ __forceinline__ void store(char *lds, const float (&r)[E][8]) const {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            uintx4 s[3];
            split3(r[e], s);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                *reinterpret_cast<uintx4 *>(lds + dst[e] + q * kPart) = s[q];
        }
    }
};

// A BM x BN tile with float32 products and sums, for the rare tile that holds
// a non-finite value: 8 k at a time through LDS, each thread its own outputs.
template <int BM, int BN, int THREADS, bool TA, bool TB>
__device__ __noinline__ void split_again(SplitGemmArgs g, int i0, int j0, char *lds) {
    constexpr int E = BM * BN / THREADS;
    float *sa = reinterpret_cast<float *>(lds), *sb = sa + 8 * BM;
    float sum[E];
#pragma unroll
    for (int e = 0; e < E; ++e) sum[e] = 0.f;
    const int j = threadIdx.x % BN, ib = threadIdx.x / BN;
    for (int k0 = 0; k0 < g.K; k0 += 8) {
        const int kn = min(8, g.K - k0);
        __syncthreads();
        for (int e = threadIdx.x; e < 8 * BM; e += THREADS) {
            const int i = min(i0 + e % BM, g.M - 1), k = e / BM;
            if (k < kn)
                sa[e] = TA ? g.a[(int64_t)(k0 + k) * g.lda + i] : g.a[(int64_t)i * g.lda + k0 + k];
        }
        for (int e = threadIdx.x; e < 8 * BN; e += THREADS) {
            const int jj = min(j0 + e % BN, g.N - 1), k = e / BN;
            if (k < kn)
                sb[e] = TB ? g.b[(int64_t)jj * g.ldb + k0 + k] : g.b[(int64_t)(k0 + k) * g.ldb + jj];
        }
        __syncthreads();
        for (int k = 0; k < kn; ++k) {
            const float y = sb[k * BN + j];
#pragma unroll
            for (int e = 0; e < E; ++e)
                sum[e] = fmaf(sa[k * BM + ib + e * (THREADS / BN)], y, sum[e]);
        }
    }
    if (j0 + j >= g.N) return;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = i0 + ib + e * (THREADS / BN);
        if (i >= g.M) continue;
        float *c = g.c + (int64_t)i * g.ldc + j0 + j;
        *c = g.beta == 0.f ? sum[e] : g.beta * *c + sum[e];
    }
}

// Origin of tile t: groups of g.group tile rows, walked column by column, so
// that a run of tiles (one XCD) touches few row and column panels.
__device__ __forceinline__ void split_tile_of(const SplitGemmArgs &g, int t, int &tm, int &tn) {
    const int per_group = g.group * g.tiles_n;
    const int gr = t / per_group, first = gr * g.group;
    const int rows = min(g.group, g.tiles_m - first);
    const int r = t - gr * per_group;
    tm = first + r % rows;
    tn = r / rows;
}

template <int BM, int BN, int BK, int WM, int WN, bool TA, bool TB>
struct SplitGemm {
    static constexpr int kThreads = (BM / WM) * (BN / WN) * 64;
    static constexpr int FM = WM / 32, FN = WN / 32;
    using At = SplitTile<BM, BK, kThreads, !TA>;
    using Bt = SplitTile<BN, BK, kThreads, TB>;
    static constexpr int kStage = At::kBytes + Bt::kBytes;
    static constexpr int kLds = 2 * kStage;

    __device__ static void run(const SplitGemmArgs &g, int t, char *lds) {
        const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
        const int wi0 = wave / (BN / WN) * WM, wj0 = wave % (BN / WN) * WN;
        int tm, tn;
        split_tile_of(g, t, tm, tn);
        const int i0 = tm * BM, j0 = tn * BN;

        At at;
        Bt bt;
        at.init(g.a, g.a_bytes, g.lda, i0, g.M, tid);
        bt.init(g.b, g.b_bytes, g.ldb, j0, g.N, tid);
        float ra[At::E][8], rb[Bt::E][8];
        floatx16 tot[FM][FN], acc[FM][FN];
        const floatx16 zero = {};
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int b = 0; b < FN; ++b) tot[a][b] = acc[a][b] = zero;

        const int full = g.K / BK, stages = (g.K + BK - 1) / BK;
        auto fetch = [&](int s) {
            const int k0 = s * BK;
            if (s < full) {
                at.template load<true>(ra, k0, BK);
                bt.template load<true>(rb, k0, BK);
            } else if (s < stages) {
                at.template load<false>(ra, k0, g.K - k0);
                bt.template load<false>(rb, k0, g.K - k0);
            }
        };
        const int ra_off = (lane >> 5) * At::kPlane + (wi0 + (lane & 31)) * 16;
        const int rb_off = At::kBytes + (lane >> 5) * Bt::kPlane + (wj0 + (lane & 31)) * 16;
        struct Frags {
            uintx4 a[FM][3], b[FN][3];
        };
        auto read = [&](const char *s, int ks, Frags &f) {
#pragma unroll
            for (int q = 2; q >= 0; --q) {
#pragma unroll
                for (int a = 0; a < FM; ++a)
                    f.a[a][q] = *reinterpret_cast<const uintx4 *>(
                        s + ra_off + q * At::kPart + ks * 2 * At::kPlane + a * 512);
#pragma unroll
                for (int b = 0; b < FN; ++b)
                    f.b[b][2 - q] = *reinterpret_cast<const uintx4 *>(
                        s + rb_off + (2 - q) * Bt::kPart + ks * 2 * Bt::kPlane + b * 512);
            }
        };
        auto mul = [&](const Frags &f) {
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int a = 0; a < FM; ++a)
#pragma unroll
                    for (int b = 0; b < FN; ++b)
                        acc[a][b] = mfma32(f.a[a][kSplitA[q]], f.b[b][kSplitB[q]], acc[a][b]);
        };
        auto compute = [&](const char *s) {
#pragma unroll
            for (int ks = 0; ks < BK / 16; ++ks) {
                Frags f;
                read(s, ks, f);
                mul(f);
            }
        };
        auto flush = [&] {
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) {
                    tot[a][b] += acc[a][b];
                    acc[a][b] = zero;
                }
        };

        fetch(0);
        at.store(lds, ra);
        bt.store(lds + At::kBytes, rb);
        __syncthreads();
        int s = 0;
        // Stages followed by a whole one: straight code.  The next stage's
        // loads are issued first and its split and LDS writes stand between
        // the matrix instructions of the second half.
        for (; s + 1 < full; ++s) {
            char *cur = lds + (s & 1) * kStage, *nxt = lds + (~s & 1) * kStage;
            at.template load<true>(ra, (s + 1) * BK, BK);
            bt.template load<true>(rb, (s + 1) * BK, BK);
            __builtin_amdgcn_sched_barrier(kSchedNoVmem);
            Frags f;
            read(cur, 0, f);
            mul(f);
            read(cur, 1, f);
            at.store(nxt, ra);
            bt.store(nxt + At::kBytes, rb);
            mul(f);
            if (s % (kSplitFlush / BK) == kSplitFlush / BK - 1) flush();
            __syncthreads();
        }
        for (; s < stages; ++s) {
            char *cur = lds + (s & 1) * kStage, *nxt = lds + (~s & 1) * kStage;
            fetch(s + 1);
            compute(cur);
            if (s + 1 < stages) {
                at.store(nxt, ra);
                bt.store(nxt + At::kBytes, rb);
            }
            if (s % (kSplitFlush / BK) == kSplitFlush / BK - 1) flush();
            __syncthreads();
        }
        flush();

        bool bad = false;
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int b = 0; b < FN; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) bad |= !__builtin_isfinite(tot[a][b][v]);
        if (__syncthreads_or(bad))
            split_again<BM, BN, kThreads, TA, TB>(g, i0, j0, lds);
        else
            put(g, i0 + wi0, j0 + wj0, lane, tot);
    }

    __device__ __forceinline__ static void put(const SplitGemmArgs &g, int i0, int j0, int lane,
                                               const floatx16 (&tot)[FM][FN]) {
#pragma unroll
        for (int b = 0; b < FN; ++b) {
            const int j = j0 + b * 32 + (lane & 31);
            if (j >= g.N) continue;
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int i = i0 + a * 32 + 8 * (v / 4) + 4 * (lane >> 5) + v % 4;
                    if (i >= g.M) continue;
                    float *c = g.c + (int64_t)i * g.ldc + j;
                    const float sum = kSplitUnscale * tot[a][b][v];
                    *c = g.beta == 0.f ? sum : g.beta * *c + sum;
                }
        }
    }
};

// The GEMM for problems of few tiles: no operand goes through LDS.  Every
// wave computes the whole BM x BN tile over its own run of k, with fragments
// loaded straight into registers a step of 16 k ahead, so nothing waits at a
// barrier; the waves' sums meet in LDS at the end, in wave order.  (Two steps
// ahead was no faster, at 1024^3 and 1001 x 1531 x 777.)
template <int BM, int BN, int WAVES, bool TA, bool TB>
struct SplitGemmRd {
    static constexpr int kThreads = WAVES * 64;
    static constexpr int FM = BM / 32, FN = BN / 32;
    static constexpr int kLds = WAVES * BM * BN * 4;
    static_assert(kLds >= 8 * (BM + BN) * 4, "split_again's tiles");

    // Rows i0 + 32 f + lane%32 of one operand, k = 8 * (lane/32) + 0..7 of a step.
    template <int F, bool KC>
    struct Frag {
        __amdgpu_buffer_rsrc_t rs;
        int off[F], ld4;
        __device__ __forceinline__ void init(const float *base, uint32_t bytes, int ld, int i0,
                                             int I, int lane) {
            rs = split_rsrc(base, bytes);
            ld4 = ld * 4;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const int row = min(i0 + f * 32 + (lane & 31), I - 1), k = (lane >> 5) * 8;
                off[f] = KC ? row * ld4 + k * 4 : k * ld4 + row * 4;
            }
        }
        // The step at k0; left: its k that exist, 16 or more with FULL.
        template <bool FULL>
        __device__ __forceinline__ void load(float (&r)[F][8], int k0, int left, int kl) const {
#pragma unroll
            for (int f = 0; f < F; ++f) {
                if constexpr (KC && FULL) {
                    load8(rs, off[f], k0 * 4, r[f]);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const bool in = FULL || kl + i < left;
                        r[f][i] = KC ? load1(rs, in ? off[f] + 4 * i : kSplitOOB, k0 * 4)
                                     : load1(rs, in ? off[f] : kSplitOOB, (k0 + i) * ld4);
                    }
                }
            }
        }
    };

    __device__ static void run(const SplitGemmArgs &g, int t, char *lds) {
        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        int tm, tn;
        split_tile_of(g, t, tm, tn);
        const int i0 = tm * BM, j0 = tn * BN;
        // Equal runs of whole steps; the last waves may have less, or none.
        const int steps_all = (g.K + 15) / 16;
        const int per = (steps_all + WAVES - 1) / WAVES;
        const int s0 = min(wave * per, steps_all), steps = min(s0 + per, steps_all) - s0;
        const int kbeg = s0 * 16, kl = (lane >> 5) * 8;

        floatx16 tot[FM][FN];
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int b = 0; b < FN; ++b) tot[a][b] = floatx16{};
        if (steps > 0) {
            Frag<FM, !TA> fa;
            Frag<FN, TB> fb;
            fa.init(g.a, g.a_bytes, g.lda, i0, g.M, lane);
            fb.init(g.b, g.b_bytes, g.ldb, j0, g.N, lane);
            float ra[FM][8], rb[FN][8];
            const int full = min(steps, (g.K - kbeg) / 16);
            auto fetch = [&](int s) {
                const int k0 = kbeg + s * 16;
                if (s < full) {
                    fa.template load<true>(ra, k0, 16, kl);
                    fb.template load<true>(rb, k0, 16, kl);
                } else if (s < steps) {
                    fa.template load<false>(ra, k0, g.K - k0, kl);
                    fb.template load<false>(rb, k0, g.K - k0, kl);
                }
            };
            fetch(0);
            floatx16 acc[FM][FN];
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) acc[a][b] = floatx16{};
            for (int s = 0; s < steps; ++s) {
                uintx4 af[FM][3], bf[FN][3];
#pragma unroll
                for (int a = 0; a < FM; ++a) split3(ra[a], af[a]);
#pragma unroll
                for (int b = 0; b < FN; ++b) split3(rb[b], bf[b]);
                fetch(s + 1);
                __builtin_amdgcn_sched_barrier(kSchedNoVmem);
#pragma unroll
                for (int q = 0; q < 6; ++q)
#pragma unroll
                    for (int a = 0; a < FM; ++a)
#pragma unroll
                        for (int b = 0; b < FN; ++b)
                            acc[a][b] = mfma32(af[a][kSplitA[q]], bf[b][kSplitB[q]], acc[a][b]);
                if (s % (kSplitFlush / 16) == kSplitFlush / 16 - 1) {
#pragma unroll
                    for (int a = 0; a < FM; ++a)
#pragma unroll
                        for (int b = 0; b < FN; ++b) {
                            tot[a][b] += acc[a][b];
                            acc[a][b] = floatx16{};
                        }
                }
            }
#pragma unroll
            for (int a = 0; a < FM; ++a)
#pragma unroll
                for (int b = 0; b < FN; ++b) tot[a][b] += acc[a][b];
        }

        float *sw = reinterpret_cast<float *>(lds) + wave * (BM * BN);
#pragma unroll
        for (int a = 0; a < FM; ++a)
#pragma unroll
            for (int b = 0; b < FN; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    sw[(a * 32 + 8 * (v / 4) + 4 * (lane >> 5) + v % 4) * BN + b * 32 +
                       (lane & 31)] = tot[a][b][v];
        __syncthreads();
        constexpr int E = BM * BN / kThreads;
        const float *s = reinterpret_cast<const float *>(lds);
        float out[E];
        bool bad = false;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            out[e] = s[tid + e * kThreads];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) out[e] += s[w * BM * BN + tid + e * kThreads];
            bad |= !__builtin_isfinite(out[e]);
            out[e] *= kSplitUnscale;
        }
        if (__syncthreads_or(bad)) {
            split_again<BM, BN, kThreads, TA, TB>(g, i0, j0, lds);
            return;
        }
        const int j = j0 + tid % BN;
        if (j >= g.N) return;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = i0 + tid / BN + e * (kThreads / BN);
            if (i >= g.M) continue;
            float *c = g.c + (int64_t)i * g.ldc + j;
            *c = g.beta == 0.f ? out[e] : g.beta * *c + out[e];
        }
    }
};

}  // namespace katsu
