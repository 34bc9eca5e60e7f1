// k_gemms.hip -- fp32 GEMM and implicit-GEMM convolution for problems with few
// output tiles (the layers of a model on one or a few images, an FC layer, a
// small GEMM) and for operands of any alignment.
//
// What bounds such a problem is the K loop of too few waves: at 64 x 64 tiles a
// 14 x 14 x 256 layer on one image is 16 workgroups, and each walks all of K at
// one LDS round trip per chunk.  Here a tile is as small as 16 x 16, so the
// tiles fill the CUs, and the W waves of a workgroup split K between them: wave
// w takes a contiguous run of 16-deep blocks, and the partial tiles are summed
// through LDS in wave order at the end.  A chain of fp32 sums grows the rounding
// error with the root of its length, so a wave adds its accumulators to its part
// of LDS every 256 k or less and starts again from zero: K split between four
// waves alone made chains of K / 4, longer than the K / 256 workgroups of the
// split-K kernel (relative error, 1 to 64 rows, K = 2048: 4.06e-7, with the folds
// 2.95e-7, split-K 2.95e-7; K = 6144: 7.0e-7, 2.95e-7, 3.0e-7).
//
// The waves share no operand, so there is no LDS staging and no barrier in the
// loop: a lane loads its MFMA operands straight from memory, D blocks ahead.
// v_mfma_f32_16x16x4f32 takes k = lane / 16 per step; with k = 4 (lane / 16) + j
// in step j a lane's A operands of a block are 16 consecutive bytes of its row,
// and with column FN (lane % 16) + j in block j of FN its B operands of one k
// are FN consecutive floats.  Lane offsets are fixed (CONV: per tap) and a block
// adds one scalar offset per operand.  The loads need 4-byte alignment only;
// rows, columns, taps and k past the operand read zeros, except that a quad
// that crosses the end of a row brings the next row's floats: columns past N
// are not stored, and the last block clears A's k past K.
//
// Measured (us, whole call; in parentheses with ACFUN_GEMMS=0: 64 x 64 tiles,
// F(2,3), or split-K with a reduce launch):
//   196 x 256 x 1024 GEMM         4.7   (14.5)    64 x 1000 x 2048 GEMM    7.0  (16.2)
//   1024^3 GEMM                  20.6   (22.7)    999 x 777 x 1333 GEMM   26.5  (57.1)
//   16 x 512 x 6144 GEMM         15.3   (19.4)    20001 x 131 x 259 GEMM  34.1  (57.2)
//   3x3 14 x 14 x 256, 1 image    7.6   (30.0)    3x3 7 x 7 x 512, 1      11.8  (60.5)
//   3x3/2 14 x 14 x 512, 1 image 12.4   (84.5)    3x3/2 28 x 28 x 256, 16 40.0  (47.1)
//   3x3 20 x 20 x 30 -> 50, 2     4.5   (21.7)    3x3 21 x 21 x 248, 1    13.1  (32.8)
//   7x7 28 x 28 x 12 -> 224, 9   28.9   (42.2)    3x3 51 x 51 x 143, 60  720    (1341)
// MFMA busy (counters): 0.47 at 1024^3, 0.41 at 999 x 777 x 1333 (208 workgroups),
// 0.05 to 0.10 in the layers of a model on one image.
#include "rt.hpp"

#include <cstdio>
#include <cstdlib>

namespace acfun {
namespace {

typedef float f4s __attribute__((ext_vector_type(4)));
typedef int i4s __attribute__((ext_vector_type(4)));
typedef int i2s __attribute__((ext_vector_type(2)));

struct GsConv {
    int H, W, Cin, KW, stride, pad, OH, OW;
    unsigned bytes;    // N*H*W*Cin*4, below 2^31
};

// FN consecutive floats per lane from rsrc at byte offset voff (per lane) +
// soff (scalar)
template <int FN>
__device__ __forceinline__ void ld(float (&d)[FN], __amdgpu_buffer_rsrc_t rsrc, unsigned voff, unsigned soff) {
    if constexpr (FN == 4) {
        const i4s v = __builtin_bit_cast(i4s, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff, soff, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = __int_as_float(v[e]);
    } else if constexpr (FN == 2) {
        const i2s v = __builtin_bit_cast(i2s, __builtin_amdgcn_raw_buffer_load_b64(rsrc, voff, soff, 0));
        d[0] = __int_as_float(v[0]);
        d[1] = __int_as_float(v[1]);
    } else {
        d[0] = __int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(rsrc, voff, soff, 0));
    }
}

// MODE GS_GEMM: a plain product.  GS_CONV: a convolution with Cin a multiple of
// 16, a block within one tap.  GS_TAPS: any Cin; K is walked as KH KW taps of
// Cin rounded up to 4 channels, so a lane's quad lies in one tap and each lane
// follows its own (kh, kw, channel).
enum { GS_GEMM, GS_CONV, GS_TAPS };
// Waves per SIMD the registers must leave room for.  Told so, the compiler keeps
// the accumulators in VGPRs; left alone it takes AGPRs and, for fold()'s VALU
// sums, a copy of each: 2 x 4 blocks then need 180 to 220 registers instead of 151
// to 166, two waves per SIMD instead of three.  A 16 x 16 tile has registers
// enough, and in VGPRs its sums move through the registers of loads to come (1 x
// 512 x 6144: 11.4 us against 10.3).
constexpr int gs_waves(int FM, int FN, int W) {
    return FM * FN >= 16 ? 2 : FM * FN >= 8 ? (W == 4 ? 3 : 2) : FN == 4 ? 4 : FN == 2 ? 5 : 1;
}
template <int FM, int FN, int W, int MODE>
__global__ __launch_bounds__(64 * W, gs_waves(FM, FN, W)) void k_gemms(const float* __restrict__ A, const float* __restrict__ B,
                                                  float* __restrict__ C, const float* __restrict__ bias,
                                                  const float* __restrict__ res, int M, int N, int K,
                                                  int lda, int ldb, int ldc, int ldr, int act, GsConv cv) {
    constexpr unsigned kOOB = 0x80000000u;
    constexpr bool CONV = MODE != GS_GEMM, TAPS = MODE == GS_TAPS;
    constexpr int TM = 16 * FM, TN = 16 * FN, LDT = TN + 4;
    constexpr int D = FM * FN >= 16 ? 2 : FM * FN >= 4 ? 3 : 4;   // 16-k blocks in flight, as registers allow
    constexpr bool REGS = FM * FN <= 4;                 // folded sums in registers; larger tiles: in LDS
    constexpr int NO = TM * TN / (64 * W) > 0 ? TM * TN / (64 * W) : 1;   // outputs per thread
    __shared__ float red[W * TM * LDT];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lg = lane >> 4;

    // XCD x = blockIdx % 8 owns a contiguous run of tiles, row tiles fastest
    const int gm = (M + TM - 1) / TM, gn = (N + TN - 1) / TN;
    const long long total = (long long)gm * gn;
    const int x = blockIdx.x & 7;
    const long long L = ((x * total) >> 3) + (blockIdx.x >> 3);
    if (L >= (((x + 1) * total) >> 3)) return;
    const int tn = (int)(L / gm), tm = (int)(L - (long long)tn * gm);
    const int m0 = tm * TM, n0 = tn * TN;

    // bias and residual of this thread's outputs, ahead of the operands
    float bv[NO], rv[NO];
#pragma unroll
    for (int o = 0; o < NO; ++o) {
        const int idx = tid + 64 * W * o, m = m0 + idx / TN, n = n0 + idx % TN;
        const bool in = idx < TM * TN && m < M && n < N;
        bv[o] = bias && in ? bias[n] : 0.f;
        rv[o] = res && in ? res[(long long)m * ldr + n] : 0.f;
    }

    const int mrows = M - m0 < TM ? M - m0 : TM;
    const __amdgpu_buffer_rsrc_t ares = CONV
        ? __builtin_amdgcn_make_buffer_rsrc((void*)A, (short)0, (int)cv.bytes, 0x00020000)
        : __builtin_amdgcn_make_buffer_rsrc((void*)(A + (long long)m0 * lda), (short)0,
                                            (int)(((mrows - 1) * lda + K) * 4), 0x00020000);
    const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)B, (short)0, (int)(((long long)(K - 1) * ldb + N) * 4), 0x00020000);

    unsigned va[FM], vb[4];
    int cbase[FM];
    unsigned long long cmask[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int m = m0 + 16 * i + lr;
        cbase[i] = 0;
        cmask[i] = 0;
        va[i] = kOOB;
        if (m < M) {
            if (CONV) {
                const int hw = cv.OH * cv.OW;
                const int n = m / hw, rem = m - n * hw;
                const int oh = rem / cv.OW, ow = rem - oh * cv.OW;
                const int ih0 = oh * cv.stride - cv.pad, iw0 = ow * cv.stride - cv.pad;
                cbase[i] = ((n * cv.H + ih0) * cv.W + iw0) * cv.Cin * 4 + (TAPS ? 0 : 16 * lg);
                unsigned rm = 0, cm = 0;
                for (int d = 0; d < 8; ++d) {
                    rm |= ((unsigned)(ih0 + d) < (unsigned)cv.H) ? (1u << d) : 0u;
                    cm |= ((unsigned)(iw0 + d) < (unsigned)cv.W) ? (1u << d) : 0u;
                }
                for (int d = 0; d < 8; ++d)
                    if ((rm >> d) & 1u) cmask[i] |= (unsigned long long)cm << (8 * d);
            } else {
                va[i] = (unsigned)((16 * i + lr) * lda + 4 * lg) * 4u;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
        vb[j] = n0 + FN * lr < N ? (unsigned)((4 * lg + j) * ldb + n0 + FN * lr) * 4u : kOOB;

    // this wave's 16-k blocks
    const int cinp = (cv.Cin + 3) & ~3, ntap = TAPS ? K / cv.Cin : 0;   // GS_TAPS: channels walked, taps
    const int nb = TAPS ? (ntap * cinp + 15) >> 4 : K >> 4;
    const int b0 = (int)((long long)wave * nb / W), n = (int)((long long)(wave + 1) * nb / W) - b0;
    // load cursor: the block's scalar offsets, CONV: its tap
    int cur = 0, ic = 0, kh = 0, kw = 0;
    unsigned sa = (unsigned)b0 * 64u, sb = (unsigned)b0 * 64u * (unsigned)ldb;
    auto set_tap = [&]() {
        const int to = (kh * cv.W + kw) * cv.Cin * 4, bit = kh * 8 + kw;
#pragma unroll
        for (int i = 0; i < FM; ++i) va[i] = (cmask[i] >> bit) & 1ull ? (unsigned)(cbase[i] + to) : kOOB;
    };
    if (TAPS) {                                         // this lane's quad of block b0
        const int k0 = 16 * b0 + 4 * lg, tap = k0 / cinp;
        ic = k0 - tap * cinp;
        kh = tap / cv.KW;
        kw = tap - kh * cv.KW;
    } else if (CONV) {
        const int k0 = 16 * b0, tap = k0 / cv.Cin;
        ic = k0 - tap * cv.Cin;
        kh = tap / cv.KW;
        kw = tap - kh * cv.KW;
        sa = (unsigned)ic * 4u;
        set_tap();
    }
    float a[D][FM][4], b[D][4][FN];
    int left[TAPS ? D : 1];                             // GS_TAPS: the quad's channels inside Cin
    const int bcol = n0 + FN * lr;
    auto load_taps = [&](float (&as)[FM][4], float (&bs)[4][FN], int& lf) {
        const int tap = kh * cv.KW + kw, bit = kh * 8 + kw;
        const int to = ((kh * cv.W + kw) * cv.Cin + ic) * 4;
        const unsigned rb = (unsigned)((tap * cv.Cin + ic) * ldb + bcol) * 4u;
        const bool in = tap < ntap;
        lf = in ? cv.Cin - ic : 0;
#pragma unroll
        for (int i = 0; i < FM; ++i)
            ld<4>(as[i], ares, in && ((cmask[i] >> (bit & 63)) & 1ull) ? (unsigned)(cbase[i] + to) : kOOB, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            ld<FN>(bs[j], bres, j < lf && bcol < N ? rb + (unsigned)(j * ldb) * 4u : kOOB, 0);
        if (cur + 1 < n) {
            ++cur;
            ic += 16;
            while (ic >= cinp) {
                ic -= cinp;
                if (++kw == cv.KW) { kw = 0; ++kh; }
            }
        }
    };
    auto load = [&](float (&as)[FM][4], float (&bs)[4][FN]) {
#pragma unroll
        for (int i = 0; i < FM; ++i) ld<4>(as[i], ares, va[i], sa);
#pragma unroll
        for (int j = 0; j < 4; ++j) ld<FN>(bs[j], bres, vb[j], sb);
        if (cur + 1 < n) {                              // past the end: the last block again
            ++cur;
            sb += 64u * (unsigned)ldb;
            sa += 64u;
            if (CONV && (ic += 16) == cv.Cin) {         // a block lies in one tap (Cin % 16 == 0)
                ic = 0;
                sa = 0;
                if (++kw == cv.KW) { kw = 0; ++kh; }
                set_tap();
            }
        }
    };
    f4s acc[FM][FN], sum[REGS ? FM : 1][REGS ? FN : 1];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            acc[i][j] = f4s{0.f, 0.f, 0.f, 0.f};
            if constexpr (REGS) sum[i][j] = acc[i][j];
        }
    // The wave's part of LDS: lane l, register e of block (i, j) <-> row
    // 16 i + 4 (l / 16) + e, column FN (l % 16) + j.  A lane meets its own elements
    // only, so adding to them needs no barrier.
    float* const rw = red + wave * (TM * LDT) + 4 * lg * LDT + FN * lr;
    bool folded = false;
    auto to_lds = [&]() {
        if (REGS || !folded) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < FN; ++j) {
                        if constexpr (REGS) rw[(16 * i + e) * LDT + j] = sum[i][j][e] + acc[i][j][e];
                        else rw[(16 * i + e) * LDT + j] = acc[i][j][e];
                    }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                asm volatile("" ::: "memory");          // a quarter at a time, as registers allow
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) rw[(16 * i + e) * LDT + j] += acc[i][j][e];
            }
        }
    };
    auto fold = [&]() {
        if constexpr (!REGS) {
            to_lds();
            folded = true;
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                if constexpr (REGS) sum[i][j] += acc[i][j];
                acc[i][j] = f4s{0.f, 0.f, 0.f, 0.f};
            }
    };
    // The wave's whole rounds of D blocks, a fold after every FOLD of them but the
    // last: with what follows it a chain is 16 blocks at most.
    constexpr int FOLD = 16 / D - 1;
    int done = 0;
    auto rounds = [&](auto round) {
        const int whole = n / D * D;
        for (;;) {
            const int stop = done + FOLD * D < whole ? done + FOLD * D : whole;
            for (; done < stop; done += D) round();
            if (done >= whole) break;
            fold();
        }
    };
    auto clear = [&](float (&as)[FM][4], int lf) {      // channels past Cin: the next pixel's floats
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) as[i][e] = e < lf ? as[i][e] : 0.f;
    };
    auto mul = [&](const float (&as)[FM][4], const float (&bs)[4][FN]) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(as[i][k], bs[k][j], acc[i][j], 0, 0, 0);
    };
    if constexpr (TAPS) {
        if (n > 0) {
            auto step = [&](float (&as)[FM][4], const float (&bs)[4][FN], int lf) {
                if (cinp != cv.Cin) clear(as, lf);
                mul(as, bs);
            };
#pragma unroll
            for (int s = 0; s < D; ++s) load_taps(a[s], b[s], left[s]);
            rounds([&]() {
#pragma unroll
                for (int s = 0; s < D; ++s) {
                    step(a[s], b[s], left[s]);
                    load_taps(a[s], b[s], left[s]);
                }
            });
#pragma unroll
            for (int s = 0; s < D - 1; ++s)
                if (done + s < n) step(a[s], b[s], left[s]);
        }
    } else if (n > 0) {
#pragma unroll
        for (int s = 0; s < D; ++s) load(a[s], b[s]);
        rounds([&]() {
#pragma unroll
            for (int s = 0; s < D; ++s) {
                mul(a[s], b[s]);
                load(a[s], b[s]);
            }
        });
#pragma unroll
        for (int s = 0; s < D - 1; ++s)
            if (done + s < n) mul(a[s], b[s]);
    }
    if (!CONV && (K & 15) && wave == W - 1) {           // K's ragged end: k past K are zeros
        const int k0 = nb * 16;
        float as[FM][4], bs[4][FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            ld<4>(as[i], ares, k0 + 4 * lg < K ? va[i] : kOOB, (unsigned)k0 * 4u);
#pragma unroll
            for (int e = 0; e < 4; ++e) as[i][e] = k0 + 4 * lg + e < K ? as[i][e] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            ld<FN>(bs[j], bres, k0 + 4 * lg + j < K ? vb[j] : kOOB, (unsigned)k0 * (unsigned)ldb * 4u);
        mul(as, bs);
    }

    to_lds();                                           // partial tiles, summed in wave order
    __syncthreads();
#pragma unroll
    for (int o = 0; o < NO; ++o) {
        const int idx = tid + 64 * W * o, row = idx / TN, col = idx % TN;
        if (idx >= TM * TN) continue;
        float v = red[row * LDT + col];
#pragma unroll
        for (int w = 1; w < W; ++w) v += red[w * (TM * LDT) + row * LDT + col];
        const int m = m0 + row, nn = n0 + col;
        if (m >= M || nn >= N) continue;
        if (bias) v = v + bv[o];
        if (res) v = v + rv[o];
        C[(long long)m * ldc + nn] = act_apply(v, act);
    }
}

// The tiles and their cost, us: fixed, then per_k * K for each tile the busiest
// CU runs (16 x 16 and 16 x 32 are bound by the vector loads, the others by MFMA
// and what latency their waves leave), and `each` for every tile after the
// first (its set-up, first loads and LDS sum).  Fitted to sweeps over M, N, K of
// ResNet-50's layers at 1 to 64 images, plain GEMMs, and convolutions of any
// channel count; within 10 % of most of them.  32 x 64 on two waves only pays
// with three or more workgroups a CU (1024^3, 512 workgroups: 36 us -- they do
// not spread over the SIMDs), and 32 x 64 on four waves (three fit on a CU) loses
// a round of workgroups past three (2000 x 999 x 333, four: 29 us against 19.5).
struct GsTile { int fm, fn, w, min_per_cu; float fixed, per_k, each; };
constexpr GsTile kGs[] = {
    {1, 1, 4, 0, 3.0f, 0.0020f, 0.5f}, {1, 2, 4, 0, 3.0f, 0.0033f, 0.55f}, {1, 4, 4, 0, 3.3f, 0.0043f, 0.75f},
    {2, 4, 4, 0, 3.8f, 0.0084f, 1.0f}, {2, 4, 2, 3, 4.0f, 0.0085f, 1.5f},  {4, 4, 8, 0, 5.0f, 0.0158f, 4.0f}};
constexpr int kGsN = sizeof(kGs) / sizeof(kGs[0]);

long long tiles_of(long long M, long long N, int bm, int bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); }

// (cus: num_cus(), a runtime call each time; one per entry of this table made the
// smallest products 0.5 us slower)
int pick(int M, int N, int K, long long cus, float* us) {
    int best = 0;
    *us = 1e30f;
    for (int i = 0; i < kGsN; ++i) {
        const GsTile& t = kGs[i];
        const long long total = tiles_of(M, N, 16 * t.fm, 16 * t.fn);
        const float n = (float)((total + cus - 1) / cus);
        const float e = t.fixed + n * t.per_k * (float)K + t.each * (n - 1.f) +
                        (t.fm == 2 && t.w == 4 && n > 3.f ? 5.f : 0.f);
        if (total >= cus * t.min_per_cu && e < *us) { *us = e; best = i; }
    }
    return best;
}

// ACFUN_GEMMS=0: never; "fm,fn,waves": that tile of kGs for every admitted shape
// (tests, sweeps).  Read once.
constexpr int kGsRule = -2, kGsOff = -1;
int gs_switch() {
    static const int v = [] {
        const char* e = getenv("ACFUN_GEMMS");
        int fm = 0, fn = 0, w = 0;
        if (!e) return kGsRule;
        if (sscanf(e, "%d,%d,%d", &fm, &fn, &w) != 3) return atoi(e) == 0 && *e ? kGsOff : kGsRule;
        for (int i = 0; i < kGsN; ++i)
            if (kGs[i].fm == fm && kGs[i].fn == fn && kGs[i].w == w) return i;
        return kGsRule;
    }();
    return v;
}

// The tile, if it beats the kernel the shape would otherwise run, else -1.  That
// kernel's time in us by the same kind of fit: k_gemm32 / k_gemm32p over
// 64 x 64 tiles (up to one per CU: 4.1 + 0.0183 K with its two K groups from
// K = 512 on; more: 0.0153 K per tile on the busiest CU, a convolution 0.0178, or 0.0169
// from two per CU on); k_gemm_f32 with split-K 16 us and little per K (so a
// K past some 6,000 on a handful of tiles stays there); k_gemm_f32 without it
// 4 us + the larger of 0.068 K and its padded product at 55 TFLOP/s (3x3 over
// 100 x 100 x 17 -> 33, 16 images: 64 us against 103 here), at 75 TFLOP/s once
// there are more than six tiles per CU and 64 columns, where its 128 x 128 tiles
// run in many rounds (3x3/2 over 83 x 65 x 16 -> 224, 33 images, 11 per CU: 55.4 us
// against 71.3; GEMM 241987 x 259 x 192: 408 against 513); with K up to 32 and 16
// rows or columns both take less than the host needs for a launch, and that is 0.2
// us less for k_gemm_f32's one argument (9 x 79 x 16: 3.6 against 3.8; 300 x 300 x
// 13, past that: 5.1 against 4.2); F(2,3) wins from
// about half a 64 x 64 tile per CU on (3x3 14 x 14 x 256: 8 images, 100 tiles,
// 21.4 against 31.4 us; 12, 148 tiles, 31.7 against 32.4 with the filter
// transform; 16, 196 tiles, 41 against 33).  A loaded model's layer has its
// transform (WINO_U: F(2,3) alone): there the unit kernel also wins with few input
// channels, one round of 32 x 64 tiles here costing 5.4 us + 0.0675 per channel
// against 4.2 to 5 + 0.085 (6 x 28 x 32 x 16 -> 48, the layer in its model: 7.6 us
// against 8.8; x 24 -> 64, 117 tiles, 9.8 against 10.4; 48 channels 11.1 against
// 11.0; 64: 13.2 against 12.3; 128: 18.7 against 16.8); with at most a quarter of
// the CUs or 32 columns smaller tiles make up for it (4 x 16 x 64 x 16 -> 32: 7.5
// against 6.9).  5 % in favour of the other kernel.
int tile_if_faster(int M, int N, int K, GsAlt alt, int Cin = 0, float scale = 1.f) {
    if (gs_switch() != kGsRule) return gs_switch();
    const long long t = tiles_of(M, N, 64, 64), cus = num_cus();
    const bool wino = alt == GsAlt::WINO || alt == GsAlt::WINO_U;
    if (wino ? 2 * t > cus : t > 2 * cus && alt != GsAlt::F32) return -1;
    if (alt == GsAlt::F32 && K <= 32 && (M <= 16 || N <= 16)) return -1;
    if (alt == GsAlt::WINO_U && 4 * t > cus && N > 32 && Cin <= 48) return -1;
    float us;
    const int tile = pick(M, N, K, cus, &us);
    if (wino) return tile;
    const float n = (float)((t + cus - 1) / cus), k = (float)K;
    float other;
    if (alt == GsAlt::SPLITK) other = 16.f + 0.0002f * k;
    else if (alt == GsAlt::F32) other = 4.f + fmaxf(0.068f * k, (float)t * k * (2.f * 64 * 64 / (t > 6 * cus && N > 64 ? 75e6f : 55e6f)));
    else if (t <= cus) other = K >= 512 ? 4.1f + 0.0183f * k : 5.5f + 0.0177f * k;
    else other = 4.2f + n * k * (alt == GsAlt::G32 ? 0.0153f : t < 2 * cus ? 0.0178f : 0.0169f);
    return us * scale < 0.95f * other ? tile : -1;
}

template <int FM, int FN, int W, int MODE>
bool launch(int M, int N, int K, const float* A, int lda, const float* B, int ldb, float* C, int ldc,
            const float* bias, int act, hipStream_t s, const float* res, int ldr, const GsConv& cv) {
    const long long total = (long long)((M + 16 * FM - 1) / (16 * FM)) * ((N + 16 * FN - 1) / (16 * FN));
    const unsigned grid = (unsigned)((total + 7) / 8 * 8);
    ACFUN_LAUNCH("k_gemms", (k_gemms<FM, FN, W, MODE>), dim3(grid), dim3(64 * W), 0, s, A, B, C, bias, res, M,
                 N, K, lda, ldb, ldc, ldr, act, cv);
    return check_launch("k_gemms");
}

template <int MODE>
bool run(int tile, int M, int N, int K, const float* A, int lda, const float* B, int ldb, float* C,
         int ldc, const float* bias, int act, hipStream_t s, const float* res, int ldr, const GsConv& cv) {
    switch (tile) {
        case 0: return launch<1, 1, 4, MODE>(M, N, K, A, lda, B, ldb, C, ldc, bias, act, s, res, ldr, cv);
        case 1: return launch<1, 2, 4, MODE>(M, N, K, A, lda, B, ldb, C, ldc, bias, act, s, res, ldr, cv);
        case 2: return launch<1, 4, 4, MODE>(M, N, K, A, lda, B, ldb, C, ldc, bias, act, s, res, ldr, cv);
        case 3: return launch<2, 4, 4, MODE>(M, N, K, A, lda, B, ldb, C, ldc, bias, act, s, res, ldr, cv);
        case 4: return launch<2, 4, 2, MODE>(M, N, K, A, lda, B, ldb, C, ldc, bias, act, s, res, ldr, cv);
        default: return launch<4, 4, 8, MODE>(M, N, K, A, lda, B, ldb, C, ldc, bias, act, s, res, ldr, cv);
    }
}

}  // namespace

int gemms_tile(int M, int N, int K, int lda, int ldb, GsAlt alt) {
    const bool fits = M > 0 && N > 0 && K > 0 && (long long)lda * 64 * 4 < 0x7fffffffll &&
           (long long)K * ldb * 4 < 0x7fffffffll && tiles_of(M, N, 16, 16) < 0x7ffffff0ll;
    return fits ? tile_if_faster(M, N, K, alt) : -1;
}

bool gemms_f32(int tile, int M, int N, int K, const float* A, int lda, const float* B, int ldb, float* C, int ldc,
               const float* bias, int act, hipStream_t s, const float* res, int ldr) {
    return run<GS_GEMM>(tile, M, N, K, A, lda, B, ldb, C, ldc, bias, act, s, res, ldr, GsConv{});
}

int convs_tile(const ConvShape& g, int Cout, GsAlt alt) {
    const long long M = (long long)g.N * g.OH * g.OW, K = (long long)g.KH * g.KW * g.Cin;
    const bool fits = M > 0 && K > 0 && Cout > 0 && g.KH <= 8 && g.KW <= 8 &&
           (long long)g.N * g.H * g.W * g.Cin * 4 < 0x7fffffffll && K * Cout * 4 < 0x7fffffffll &&
           M < 0x7fffffffll && tiles_of(M, Cout, 16, 16) < 0x7ffffff0ll;
    // GS_TAPS: address work per block
    return fits ? tile_if_faster((int)M, Cout, (int)K, alt, g.Cin, g.Cin % 16 ? 1.25f : 1.f) : -1;
}

bool convs_f32(int tile, const ConvShape& g, const float* in, const float* w, const float* bias, int Cout, float* out,
               int act, hipStream_t s, const float* res, int ldr) {
    const GsConv cv{g.H, g.W, g.Cin, g.KW, g.stride, g.pad, g.OH, g.OW,
                    (unsigned)((long long)g.N * g.H * g.W * g.Cin * 4)};
    const int M = g.N * g.OH * g.OW, K = g.KH * g.KW * g.Cin;
    if (g.Cin % 16 == 0)
        return run<GS_CONV>(tile, M, Cout, K, in, g.Cin, w, Cout, out, Cout, bias, act, s, res, ldr, cv);
    return run<GS_TAPS>(tile, M, Cout, K, in, g.Cin, w, Cout, out, Cout, bias, act, s, res, ldr, cv);
}

}  // namespace acfun
