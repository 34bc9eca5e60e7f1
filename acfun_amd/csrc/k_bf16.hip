// k_bf16.hip -- acfun_gemm_bf16 on bf16 MFMA.
//
// Replaces the reference's AVX-512 BF16 path (src/gemm_bf16_avx512.cpp): A and
// B are rounded to bf16 (round to nearest even on bit 16, :37-44) and the
// products accumulate in fp32.  Products of two bf16 values are exact in fp32,
// so the result differs from the reference only by the fp32 accumulation
// order.
//
// One packing launch writes the rounded operands k-contiguous -- A as
// [M][Kp], B transposed as [N][Kp], Kp = K rounded up to 128, zeros beyond K
// -- and k_bf16mm multiplies them on v_mfma_f32_32x32x16_bf16.
//
// k_bf16mm: WM x WN waves, each FM x FN accumulators of 32 x 32; K in chunks
// of KB bytes DMA'd into LDS by buffer_load_dwordx4 ... lds (lane offsets fixed,
// one scalar offset per chunk), NST stages.  In k-step s of a chunk lane half h
// reads quad 2s + h of its A rows and B rows: eight bf16 each, the MFMA's 16 k.
// A k-step's operands are read while the step before is multiplied, and the
// last step's MFMAs cover the barrier and the first reads of the next chunk
// (64 x 64 tiles, one MFMA per step, read the whole chunk up front).
//
// What bounds a large product with small tiles is LDS: a wave of FM x FN blocks
// reads 32 (FM + FN) bytes per lane pair for FM x FN MFMAs, and with 64 x 64 tiles
// (FM = FN = 1) that and the DMA writes take four times the MFMA time.  256 x 256
// tiles on eight 128 x 64 waves bring LDS down to about the MFMA time, at one
// workgroup per CU; they need 256 tiles to fill the chip.  There neither fills the
// time alone (4096^3: MFMA busy 0.59, LDS reads 0.44 of the cycles, half of them
// counted as bank conflicts, and the DMA's writes on top).  Measured, us for
// k_bf16mm alone with 64 x 64 / 128 x 128 / 256 x 256:
//   4096^3              289 / 127 / 111 (1,234 TFLOP/s)
//   3008 x 2000 x 4096  109 /  54 /  81
//   2048^3               41 /  21 /  44
//   1024^3              6.9 / 11.9 / 25
// A whole 4096^3 call, the packing launch (31 us) included, takes 142 to 149 us back
// to back and 152 with other operands each time; with 64 x 64 tiles 330 and 339.
#include "rt.hpp"

namespace acfun {
namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef int i4v __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;

// fp32 -> bf16 bits as the reference packs its operands
// (src/gemm_bf16_avx512.cpp:37-44): add 0x7fff plus bit 16, keep the upper
// half.  The 32-bit add wraps, so some NaNs become infinities or zero there
// too.
__device__ __forceinline__ unsigned bf16_bits(float f) {
    const unsigned u = __float_as_uint(f);
    return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
}

// One lane: 8 consecutive k of one row of A -> one 16-byte store (two 16-byte
// loads when the row segment is whole and aligned).
__device__ __forceinline__ void pack_a_bf16(long long t, const float* __restrict__ A, int M, int K,
                                            int lda, unsigned short* __restrict__ Ab, int Kp, bool va) {
    const int kq = Kp >> 3;
    if (t >= (long long)M * kq) return;
    const int m = (int)(t / kq), k0 = (int)(t - (long long)m * kq) * 8;
    const float* src = A + (long long)m * lda + k0;
    float v[8];
    if (va && k0 + 8 <= K) {
        const float4 x0 = *(const float4*)src, x1 = *(const float4*)(src + 4);
        v[0] = x0.x; v[1] = x0.y; v[2] = x0.z; v[3] = x0.w;
        v[4] = x1.x; v[5] = x1.y; v[6] = x1.z; v[7] = x1.w;
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = k0 + e < K ? src[e] : 0.f;
    }
    unsigned w[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const unsigned lo = k0 + 2 * p < K ? bf16_bits(v[2 * p]) : 0u;
        const unsigned hi = k0 + 2 * p + 1 < K ? bf16_bits(v[2 * p + 1]) : 0u;
        w[p] = lo | (hi << 16);
    }
    *(i4v*)(Ab + (long long)m * Kp + k0) = i4v{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
}

// One block: a 64 k x 64 n tile of B -> Bt[n][k] through LDS.  Thread t loads
// quad t % 16 of rows t / 16 + 16 i (256 contiguous bytes per row), rounds
// each value (the same bf16_bits) and writes it transposed into LDS; then 8
// threads store the 128 bytes of one Bt row segment (16 bytes each).  k past K
// is zero (Kp padding); n past N is not stored.
__device__ __forceinline__ void pack_bt_bf16(int tile, const float* __restrict__ B, int K, int N, int ldb,
                                             unsigned short* __restrict__ Bt, int Kp, bool vb) {
    __shared__ unsigned short tr[64][64 + 8];          // [n][k], rows padded by 16 bytes
    const int t = (int)threadIdx.x;
    const int ntn = (N + 63) >> 6;
    const int kb = tile / ntn, nb = tile - kb * ntn;
    const int k0 = kb * 64, n0 = nb * 64;
    const int q = t & 15, n = n0 + 4 * q;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int kr = (t >> 4) + 16 * i, k = k0 + kr;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        if (k < K) {
            const float* src = B + (long long)k * ldb + n;
            if (vb && n + 4 <= N) {
                const float4 x = *(const float4*)src;
                v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = n + e < N ? src[e] : 0.f;
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) tr[4 * q + e][kr] = k < K ? (unsigned short)bf16_bits(v[e]) : (unsigned short)0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int nr = (t >> 3) + 32 * i, kc = 8 * (t & 7);
        if (n0 + nr < N && k0 + kc < Kp)
            *(i4v*)(Bt + (long long)(n0 + nr) * Kp + k0 + kc) = *(const i4v*)&tr[nr][kc];
    }
}

// Both operands in one launch: blocks [0, nba) pack A (8 k per lane), the
// rest B (a 64 x 64 tile per block).
__global__ __launch_bounds__(256) void k_pack_bf16(const float* __restrict__ A, const float* __restrict__ B,
                                                   int M, int N, int K, int lda, int ldb, int Kp, int nba,
                                                   unsigned short* __restrict__ Ab,
                                                   unsigned short* __restrict__ Bt, int va, int vb) {
    const int b = (int)blockIdx.x;
    if (b < nba) pack_a_bf16((long long)b * 256 + threadIdx.x, A, M, K, lda, Ab, Kp, va != 0);
    else pack_bt_bf16(b - nba, B, K, N, ldb, Bt, Kp, vb != 0);
}

// s_waitcnt vmcnt(n), n < 64
constexpr int bf_vmcnt(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }

__device__ __forceinline__ void bf_dma16(__amdgpu_buffer_rsrc_t rsrc, char* lds, unsigned voff, unsigned soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)lds, 16, voff, soff, 0, 0);
}

template <int WM, int WN, int FM, int FN, int KB, int NST>
struct BfTile {
    static constexpr int BM = 32 * WM * FM, BN = 32 * WN * FN, T = 64 * WM * WN;
    static constexpr int SA = BM * KB, STG = (BM + BN) * KB, LDS = NST * STG;
};

template <int WM, int WN, int FM, int FN, int KB, int NST>
__global__ __launch_bounds__(64 * WM * WN) void k_bf16mm(const unsigned short* __restrict__ Ab,
                                                         const unsigned short* __restrict__ Bt,
                                                         float* __restrict__ C, int M, int N, int Kp,
                                                         int ldc, unsigned a_bytes, unsigned b_bytes) {
    using Tl = BfTile<WM, WN, FM, FN, KB, NST>;
    constexpr int BM = Tl::BM, BN = Tl::BN, NW = WM * WN;
    constexpr int QR = KB / 16, RPI = 64 / QR;          // quads per row, rows per DMA instruction
    constexpr int AIT = BM / RPI / NW, BIT = BN / RPI / NW, ITEMS = AIT + BIT;
    constexpr int KS = KB / 32;                         // k-steps of 16 per chunk
    constexpr unsigned kOOB = 0x80000000u;
    static_assert(AIT * RPI * NW == BM && BIT * RPI * NW == BN, "whole DMA instructions per wave");
    static_assert(KS % 2 == 0 && NST >= 2 && (NST - 1) * ITEMS < 64, "operand sets, vmcnt");
    extern __shared__ __attribute__((aligned(16))) char smb[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave - wm * WN;
    // XCD x (workgroup id mod 8) owns a contiguous run of tiles; a run goes in
    // groups of 4 tile rows, column-major inside, so the tiles an XCD runs
    // together are a compact patch whose operands share its L2
    const int gn = (N + BN - 1) / BN, gm = (M + BM - 1) / BM, total = gn * gm;
    const int x = blockIdx.x & 7;
    const int L = (int)(((long long)x * total) >> 3) + (int)(blockIdx.x >> 3);
    if (L >= (int)(((long long)(x + 1) * total) >> 3)) return;
    constexpr int GRP = 4;
    const int grp = L / (GRP * gn), rows = gm - grp * GRP < GRP ? gm - grp * GRP : GRP;
    const int rin = L - grp * GRP * gn;
    const int m0 = (grp * GRP + rin % rows) * BM, n0 = (rin / rows) * BN;
    const int nch = Kp / (KB / 2);
    // quad q of row r sits at slot q ^ sw(r): 8 consecutive rows' reads of one
    // quad take 8 different slots
    auto sw = [](int r) { return QR >= 8 ? r & (QR - 1) : (r >> 1) & (QR - 1); };
    const int sl = lane % QR, rl = lane / QR;
    unsigned av[AIT], bv[BIT];
#pragma unroll
    for (int t = 0; t < AIT; ++t) {
        const int row = RPI * (wave + NW * t) + rl, q = sl ^ sw(row);
        av[t] = m0 + row < M ? (unsigned)((m0 + row) * Kp * 2 + 16 * q) : kOOB;
    }
#pragma unroll
    for (int t = 0; t < BIT; ++t) {
        const int row = RPI * (wave + NW * t) + rl, q = sl ^ sw(row);
        bv[t] = n0 + row < N ? (unsigned)((n0 + row) * Kp * 2 + 16 * q) : kOOB;
    }
    // Every iteration issues one chunk, so all waits of the loop are the same; past
    // the last one out of range (an empty buffer): no memory traffic, and zeros to
    // a stage whose contents are not multiplied.
    auto issue = [&](int c, char* st) {
        const bool live = c < nch;
        const unsigned so = live ? (unsigned)c * KB : 0u;
        const __amdgpu_buffer_rsrc_t ares =
            __builtin_amdgcn_make_buffer_rsrc((void*)Ab, (short)0, live ? (int)a_bytes : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t bres =
            __builtin_amdgcn_make_buffer_rsrc((void*)Bt, (short)0, live ? (int)b_bytes : 0, 0x00020000);
#pragma unroll
        for (int t = 0; t < AIT; ++t) bf_dma16(ares, st + (wave + NW * t) * 1024, av[t], so);
#pragma unroll
        for (int t = 0; t < BIT; ++t) bf_dma16(bres, st + Tl::SA + (wave + NW * t) * 1024, bv[t], so);
    };
    // LDS read offsets of k-step s: a lane's quad 2 s + h of its rows
    const int r32 = lane & 31, hq = lane >> 5;
    const int ra = wm * 32 * FM + r32, rb = wn * 32 * FN + r32;     // + 32 i: the same swizzle
    int qo[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) qo[s] = 16 * ((2 * s + hq) ^ sw(r32));
    f16v acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    auto read = [&](i4v (&a)[FM], i4v (&b)[FN], const char* S, int s) {
#pragma unroll
        for (int i = 0; i < FM; ++i) a[i] = *(const i4v*)(S + (ra + 32 * i) * KB + qo[s]);
#pragma unroll
        for (int j = 0; j < FN; ++j) b[j] = *(const i4v*)(S + Tl::SA + (rb + 32 * j) * KB + qo[s]);
    };
    auto mul = [&](const i4v (&a)[FM], const i4v (&b)[FN]) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    __builtin_bit_cast(bf8, a[i]), __builtin_bit_cast(bf8, b[j]), acc[i][j], 0, 0, 0);
    };
    if constexpr (FM * FN == 1) {
        // one MFMA per k-step hides nothing: all of a chunk's reads up front
        constexpr int AHEAD = NST - 1;
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) issue(a, smb + a * Tl::STG);
        int st = 0;
        for (int c = 0; c < nch; ++c) {
            // chunk c landed (the AHEAD - 1 chunks after it stay in flight), and
            // every wave has read chunk c - 1, whose stage chunk c + AHEAD takes
            __builtin_amdgcn_s_waitcnt(bf_vmcnt((AHEAD - 1) * ITEMS));
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            i4v ca[KS][FM], cb[KS][FN];
#pragma unroll
            for (int s = 0; s < KS; ++s) read(ca[s], cb[s], smb + st * Tl::STG, s);
            issue(c + AHEAD, smb + (st == 0 ? NST - 1 : st - 1) * Tl::STG);
#pragma unroll
            for (int s = 0; s < KS; ++s) mul(ca[s], cb[s]);
            st = st == NST - 1 ? 0 : st + 1;
        }
    } else {
        i4v fa[2][FM], fb[2][FN];                       // a k-step's operands, one step ahead
#pragma unroll
        for (int a = 0; a < NST; ++a) issue(a, smb + a * Tl::STG);
        __builtin_amdgcn_s_waitcnt(bf_vmcnt((NST - 1) * ITEMS));
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        read(fa[0], fb[0], smb, 0);
        int st = 0;
        for (int c = 0; c < nch; ++c) {
            char* const S = smb + st * Tl::STG;
#pragma unroll
            for (int s = 0; s < KS - 1; ++s) {
                read(fa[(s + 1) & 1], fb[(s + 1) & 1], S, s + 1);
                __builtin_amdgcn_sched_barrier(0);          // the next step's reads before this one's MFMAs
                mul(fa[s & 1], fb[s & 1]);
            }
            // chunk c is in registers (everyone's): its stage takes chunk c + NST.
            // Chunk c + 1 has landed once the NST - 2 chunks after it are all that
            // is outstanding; the last step's MFMAs cover its first reads.
            __builtin_amdgcn_s_waitcnt(bf_vmcnt((NST - 2) * ITEMS));
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            st = st == NST - 1 ? 0 : st + 1;
            read(fa[0], fb[0], smb + st * Tl::STG, 0);
            issue(c + NST, S);
            __builtin_amdgcn_sched_barrier(0);
            mul(fa[(KS - 1) & 1], fb[(KS - 1) & 1]);
        }
    }
    // epilogue: lane l, register e of block (i, j) <-> row 32 i + 8 (e / 4) +
    // 4 (l / 32) + e % 4, column 32 j + l % 32 of the wave's part
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int n = n0 + (wn * FN + j) * 32 + r32;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = m0 + (wm * FM + i) * 32 + 8 * (e >> 2) + 4 * hq + (e & 3);
                if (m < M && n < N) C[(long long)m * ldc + n] = acc[i][j][e];
            }
        }
    __builtin_amdgcn_s_waitcnt(bf_vmcnt(0));            // the chunks issued past the end, still on their way to LDS
}

template <int WM, int WN, int FM, int FN, int KB, int NST>
bool launch_bf16(const unsigned short* Ab, const unsigned short* Bt, float* C, int M, int N, int Kp, int ldc,
                 hipStream_t s) {
    using Tl = BfTile<WM, WN, FM, FN, KB, NST>;
    static_assert(Tl::LDS <= 160 * 1024, "LDS");
    // set once per process, thread-safely, before any launch below
    static const bool attr = [] {
        (void)hipFuncSetAttribute((const void*)k_bf16mm<WM, WN, FM, FN, KB, NST>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, Tl::LDS);
        return true;
    }();
    (void)attr;
    const long long tiles = (long long)((M + Tl::BM - 1) / Tl::BM) * ((N + Tl::BN - 1) / Tl::BN);
    ACFUN_LAUNCH("k_bf16mm", (k_bf16mm<WM, WN, FM, FN, KB, NST>), dim3((unsigned)((tiles + 7) / 8 * 8)),
                 dim3(Tl::T), Tl::LDS, s, Ab, Bt, C, M, N, Kp, ldc, (unsigned)((long long)M * Kp * 2),
                 (unsigned)((long long)N * Kp * 2));
    return check_launch("k_bf16mm");
}

// C[0:M, 0:N] (row stride ldb = ldc) = bf16(A[0:M, :]) x bf16(B[:, 0:N]) on bf16 MFMA
bool bf16_region(int M, int N, int ldb, int K, const float* A, const float* B, float* C,
                 hipStream_t s) {
    const int Kp = (K + 127) / 128 * 128;
    if ((long long)M * Kp * 2 >= 0x7fffffffll || (long long)N * Kp * 2 >= 0x7fffffffll) {
        set_error("acfun_gemm_bf16: operands beyond 2 GB");
        return false;
    }
    Scratch ab((size_t)M * Kp * 2, s), bt((size_t)N * Kp * 2, s);
    if (!ab.p || !bt.p) return false;
    const long long na = (long long)M * (Kp / 8);
    const long long nba = (na + 255) / 256, nbb = (long long)(Kp / 64) * ((N + 63) / 64);
    if (nba + nbb >= (1ll << 31)) {
        set_error("acfun_gemm_bf16: operands too large");
        return false;
    }
    auto al = [](const void* p) { return ((uintptr_t)p & 15u) == 0; };
    const int va = al(A) && K % 4 == 0, vb = al(B) && ldb % 4 == 0 && N % 4 == 0;
    ACFUN_LAUNCH("k_pack_bf16", k_pack_bf16, dim3((unsigned)(nba + nbb)), dim3(256), 0, s, A, B, M, N, K, K, ldb, Kp,
                       (int)nba, ab.as<unsigned short>(), bt.as<unsigned short>(), va, vb);
    if (!check_launch("k_pack_bf16")) return false;
    const unsigned short *pa = ab.as<unsigned short>(), *pb = bt.as<unsigned short>();
    // Tile by the time of the busiest CU, us, fitted to the sizes above: a tile
    // costs 0.0040, 0.0090 alone on its CU (eight waves, three stages) or 0.0075
    // beside another (four waves, two workgroups per CU), and 0.0262 per K.
    const long long cus = num_cus();
    auto per_cu = [&](int b) {
        const long long t = (long long)((M + b - 1) / b) * ((N + b - 1) / b);
        return (float)((t + cus - 1) / cus);
    };
    const float n128 = per_cu(128), k = (float)Kp;
    const float t64 = 3.f + per_cu(64) * k * 0.0040f;
    const float t128 = 3.f + (n128 < 2.f ? k * 0.0090f : n128 * k * 0.0075f);
    const float t256 = 4.f + per_cu(256) * k * 0.0262f;
    if (t256 < t128 && t256 < t64) return launch_bf16<2, 4, 4, 2, 128, 2>(pa, pb, C, M, N, Kp, ldb, s);
    if (t64 <= t128) return launch_bf16<2, 2, 1, 1, 256, 4>(pa, pb, C, M, N, Kp, ldb, s);
    if (n128 < 2.f) return launch_bf16<2, 4, 2, 1, 128, 3>(pa, pb, C, M, N, Kp, ldb, s);
    return launch_bf16<2, 2, 2, 2, 128, 2>(pa, pb, C, M, N, Kp, ldb, s);
}

}  // namespace

// The reference's split (src/gemm_bf16_avx512.cpp:123-168): its 16 x 16
// micro-tiles multiply bf16-rounded operands; the rows past the last multiple
// of 16 of M and the columns past the last multiple of 16 of N (its 256 x 128
// tiles are multiples of 16) take the scalar fp32 path on the unrounded
// operands.  Here k_bf16mm covers the first region and the fp32 GEMM engine
// the two strips.  K <= 0 leaves C untouched, as there (:173).
bool gemm_bf16_dev(int M, int N, int K, const float* A, const float* B, float* C, hipStream_t s) {
    if (M <= 0 || N <= 0 || K <= 0) return true;
    const int M16 = M / 16 * 16, N16 = N / 16 * 16;
    if (M16 < M && !gemm_f32(M - M16, N, K, A + (long long)M16 * K, K, B, N, C + (long long)M16 * N, N,
                             nullptr, 0, s))
        return false;
    if (N16 < N && M16 > 0 && !gemm_f32(M16, N - N16, K, A, K, B + N16, N, C + N16, N, nullptr, 0, s))
        return false;
    if (M16 == 0 || N16 == 0) return true;
    return bf16_region(M16, N16, N, K, A, B, C, s);
}

}  // namespace acfun
