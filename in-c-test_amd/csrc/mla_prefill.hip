// HIP kernels of the causal MLA prefill (src/mla_prefill_streaming.c:78-206 of the
// reference: non-absorbed attention, K/V expanded through kv_b for every token).
//
// MFMA route (H, R and NH * DV multiples of 64, QD = 192, DV = 128, DN multiple of 8):
//   split     x (fp32) -> bf16 hi + lo operands; a flag records whether any lo is non-zero (a short
//             prompt without a state fill skips this: its projection splits fp32 x itself)
//   gemm      [q | kv_a] = x . W^T           (bf16 MFMA, fp32 accumulate, the lo part skipped
//                                             when the operand is exactly bf16); epilogue:
//                                             Q = [q_nope | RoPE(q_rope)] as fp16 hi and bf8 lo.
//   kva_pack  RMSNorm -> latent (hi/lo bf16), RoPE(k_rope) -> rope part of K (fp16 hi + K8)
//   gemm      kv = latent . kv_b^T           epilogue: k_nope -> K (fp16 hi + K8), V^T (fp16)
//   flash     causal attention per (64- or 128-query tile, head), online softmax; scores Kh Qh in
//             fp16 plus the Kh Ql + Kl Qh correction from bf8 operands (K8: bf8 of the hi
//             parts and of the lo parts x 2^11)
//   gemm      out = heads . o_proj^T          (fp16 heads and fp16 copy of o_proj, one pass)
// Generic route (any shape): the same stages with VALU kernels.
//
// Range of the 16-bit operands. V (and so the attention output) and the fp16 o_proj copy carry
// power-of-two scales chosen by the host from bounds it knows (|V| <= sqrt(R) max|norm weight|
// max ||kv_b row||_2; max|o_proj|), undone exactly by the o_proj epilogue. Q and K depend on x
// and are not scaled; the flash kernel checks every query row instead: a row whose reference
// max logit exceeds kFLogitMax (beyond it the bf8 score correction's error grows past the 2e-3
// budget) or whose output is not finite raises a per-call flag (and a sticky flag for callers
// that read it later). The o_proj epilogue then writes NaN, and the host-buffer entry points
// run the call again on the generic route.
#include "mla_device.h"
#include "mla_internal.h"

#include <math.h>

#include <algorithm>
#include <type_traits>

namespace kvl {

// ================================================================ split ================

// src[r, c] (fp32, ld_src) -> hi/lo bf16 [rows, cols] (ld_dst); flag |= any lo != 0.
// Each thread converts 8 consecutive values (cols % 8 == 0, 16-byte aligned rows).
__global__ __launch_bounds__(256) void k_split(const float *src, int ld_src, uint16_t *hi,
                                               uint16_t *lo, int ld_dst, int rows, int cols,
                                               int *flag) {
    const int c8 = cols / 8;
    int any = 0;
    // flag[1]: the range flag of this call (raised by the flash kernel, read by the o_proj
    // epilogue), cleared here, in the call's first kernel
    if (flag && blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(flag + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    // rows over blocks, 8-column groups over threads (no index division in the loop)
    for (int r = blockIdx.x; r < rows; r += gridDim.x) {
        const float *s = src + (size_t)r * ld_src;
        uint16_t *hr = hi + (size_t)r * ld_dst, *lr = lo + (size_t)r * ld_dst;
        for (int c = 8 * threadIdx.x; c < 8 * c8; c += 8 * 256) {
            const v4f x0 = *(const v4f *)(s + c), x1 = *(const v4f *)(s + c + 4);
            v8bf h, l;
            split8(x0, x1, h, l);
            *(v8bf *)(hr + c) = h;
            *(v8bf *)(lr + c) = l;
            const v4i lv = __builtin_bit_cast(v4i, l);
            any |= ((lv.x | lv.y | lv.z | lv.w) & 0x7fff7fff) != 0;
        }
    }
    // Blocks with a non-zero lo word store 1. Every writer stores the same value and the reader
    // is a later kernel, so a workgroup-scope store (cached in the XCD's L2, written back at
    // the kernel's end) suffices; device-coherent stores or atomics to one address from every
    // block serialise at memory (measured 13-65 us for 2048 blocks). The flag is only raised
    // here; k_kva_pack clears it after the q GEMM has read it.
    if (flag && __syncthreads_or(any) && threadIdx.x == 0)
        __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// ================================================================ GEMM =================

// C[m, n] = sum_k (Ah + Al)[m, k] * B[n, k]: row-major bf16 operands, fp32 output. The
// columns of C may come from two weight matrices (B0 for n < N0, B1 for the N1 after it),
// so the q and kv_a projections of the same tokens run as one launch.
//
// Block tile BM x BN, MW math waves in a WM x WN grid, each owning (BM / WM) x 16 TN columns of
// v_mfma_f32_16x16x32 tiles. With LO a stage of the LDS ring holds a k step of Ah, of Al and of
// B, so each B tile is taken in once for both parts (two passes over k took in 4/3 of the
// bytes); the Al part is neither fetched nor multiplied when *lo_flag says that it is zero.
// The stages stream in by global_load_lds_dwordx4 DMA, issued by four more waves that do nothing
// else: a DMA instruction holds its wave until the memory system accepts it (about a quarter of
// a math wave's time when the math waves issued their own), so the math waves only compute and
// meet the DMA waves at one barrier per stage (the DMA waves wait for stage kt's data before it).
// The 16-byte slots of a row are XOR-swizzled so that the 8 rows one ds_read_b128 phase touches
// fall into distinct banks. Each wave reads all its fragments of a 32-deep k-sub before its
// MFMAs. The lo part runs when Al is given and either no flag is given or *lo_flag != 0 (the
// flag is raised by the producer of Al when some lo word is non-zero). Requires K % 64 == 0, lda
// and ldb multiples of 8.
constexpr int kGemmDma = 4;  // DMA waves of a GEMM block

// AF32 (with LO): A comes as fp32 (GemmArgs::Af) and the math waves split it (split8_cvt, the words
// k_split makes of finite values): the bytes of the two planes, without the launch that writes them.
template <int BM_, int BN_, int BK_, int MW_, int BPC_, bool LO_, bool AF32_ = false>
struct GemmCfg {
    static constexpr int BM = BM_, BN = BN_, BK = BK_, MW = MW_, BPC = BPC_;  // BPC: blocks per CU
    static constexpr bool LO = LO_, AF32 = AF32_;
    static constexpr int RowB = BK * 2, Spr = BK / 8;  // 16-byte slots per row
    static constexpr int TN = BN >= 64 ? 4 : BN / 16;  // 16-column tiles per wave
    static constexpr int WN = BN / (16 * TN), WM = MW / WN, TM = BM / WM / 16;
    static constexpr int ATile = BM * RowB, BTile = BN * RowB;
    static constexpr int Stage = (LO ? 2 : 1) * ATile + BTile;  // A hi, B, A lo; AF32: A, B
    static constexpr int BOff = (AF32 ? 2 : 1) * ATile, ALo = ATile + BTile;
    static constexpr int Fit = (160 * 1024 / BPC) / Stage;
    static constexpr int Stages = Fit > 8 ? 8 : Fit;  // ring depth that fits
    static constexpr int Smem = Stages * Stage;
    static constexpr int Threads = 64 * (MW + kGemmDma);
    static_assert(LO || !AF32, "fp32 A is split into hi and lo");
    static_assert(Stages >= 2 && TM >= 1 && WM * WN == MW && WM * TM * 16 == BM, "tile shape");
    static_assert(Smem >= MW * 16 * (16 * TN + 4) * 4, "the epilogue's staging fits the ring");
    __device__ static int swz(int row) { return BK == 64 ? row & 7 : (row >> 1) & 3; }
};

struct GemmArgs {
    const uint16_t *Ah, *Al, *B0, *B1;
    float *C;
    const int *lo_flag;
    int M, N0, N1, K, lda, ldb, ldc;
    const float *Af;  // fp32 A [M, lda] (GemmCfg::AF32)
    int *clear;       // a word the launch clears (may be null)
};

// Epilogues. kEpiPlain: C fp32. kEpiQ (q | kv_a projection): the N0 = NH * QD q columns go
// to Q [NH, Sp, QD] as hi/lo fp16 with the rope half rotated (src/mla_prefill_streaming.c:
// 139-147: pairs (2i, 2i+1) -> i and DR/2 + i), the kv_a columns to C (ldc = N1). kEpiKV
// (kv_b projection): k_nope -> K hi [NH, Sp, QD] fp16 and K8 [NH, Sp, 384 bytes] (bf8 of the
// hi parts and of the lo parts x 2^11, k8_hi_byte order), values -> V^T [NH, DV, Sp] fp16 with
// the keys of each 32-key group in vt_perm order.
enum { kEpiPlain = 0, kEpiQ = 1, kEpiKV = 2 };
struct GemmEpi {
    _Float16 *qh, *kh;
    uint8_t *ql8;  // bf8(Q lo x 2^11), the flash kernel's correction operand (kEpiQ)
    uint8_t *k8;
    _Float16 *vt;
    const float2 *cs;
    int Sp, DN, DR, DV;
    float vscale = 1.0f;             // kEpiKV: V^T = vscale * v (a power of two)
    float alpha = 1.0f;              // kEpiPlain: C = alpha * acc (a power of two)
    const int *nan_flag = nullptr;   // kEpiPlain: C = NaN when *nan_flag != 0
};

// Columns nl0 .. nl0 + 3 (nl0 % 4 == 0) of token t of the q projection into Q (kEpiQ). Q (50 MB at
// 4096 tokens) is read once, by the flash kernel's workgroup of its query tile: non-temporal stores
// keep it from evicting the K/V and weight lines the next kernels reuse (q GEMM 78 -> 70 us, kv_b
// GEMM 44 -> 40 us). Q hi as fp16 and Q lo only as the bf8 byte the flash kernel's correction takes
// (bf8(lo x 2^11)): 37.5 instead of 50 MB written at 4096 tokens.
__device__ __forceinline__ void store_q4(const GemmEpi &e, int t, int nl0, const v4f &x) {
    const int QD = e.DN + e.DR, half = e.DR / 2;
    const int h = nl0 / QD, k0 = nl0 % QD;
    const size_t o = ((size_t)h * e.Sp + t) * QD;
    if (k0 < e.DN) {
        v4h hi, lo;
        split4_f16(x, hi, lo);
        __builtin_nontemporal_store(hi, (v4h *)(e.qh + o + k0));
        __builtin_nontemporal_store(bf8_lo_s11(lo), (uint32_t *)(e.ql8 + o + k0));
        return;
    }
    // pairs (x.x, x.y), (x.z, x.w) of rope indices i2, i2 + 1
    const int i2 = (k0 - e.DN) >> 1;
    const float2 *cs = e.cs + (size_t)t * half + i2;
    const float2 c0 = cs[0], c1 = cs[1];
    const v4f r = {x.x * c0.x - x.y * c0.y, x.z * c1.x - x.w * c1.y, x.y * c0.x + x.x * c0.y, x.w * c1.x + x.z * c1.y};
    v4h hi, lo;
    split4_f16(r, hi, lo);
    const uint32_t l8 = bf8_lo_s11(lo);
    __builtin_nontemporal_store(__builtin_shufflevector(hi, hi, 0, 1), (v2h *)(e.qh + o + e.DN + i2));
    __builtin_nontemporal_store((uint16_t)l8, (uint16_t *)(e.ql8 + o + e.DN + i2));
    __builtin_nontemporal_store(__builtin_shufflevector(hi, hi, 2, 3), (v2h *)(e.qh + o + e.DN + half + i2));
    __builtin_nontemporal_store((uint16_t)(l8 >> 16), (uint16_t *)(e.ql8 + o + e.DN + half + i2));
}

// Position of key k (0..31 within its 32-key group) in the permuted V^T rows: the 8 keys
// lane group g of the flash kernel holds for one PV chunk are 4g .. 4g+3 and 16+4g .. 16+4g+3.
__host__ __device__ __forceinline__ int vt_perm(int k) { return 8 * ((k & 15) >> 2) + 4 * (k >> 4) + (k & 3); }

// F16: the 16-bit operands are fp16 (v_mfma_f32_16x16x32_f16) instead of bf16.
template <bool F16>
__device__ __forceinline__ v4f mfma16(const v8bf &a, const v8bf &b, const v4f &c) {
    if constexpr (F16) return mfma_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c);
    else return mfma_bf16(a, b, c);
}

// s_waitcnt vmcnt(PER * min(later, MAXL)) for a wave-uniform count of later stages in flight.
template <int PER, int MAXL>
__device__ __forceinline__ void wait_stages(int later) {
    if constexpr (MAXL == 0) {
        wait_vmcnt<0>();
    } else {
        if (later >= MAXL) wait_vmcnt<PER * MAXL>();
        else wait_stages<PER, MAXL - 1>(later);
    }
}

template <class Sh, int EPI, bool F16>
__global__ __launch_bounds__(Sh::Threads, (Sh::MW + kGemmDma) / 4 * Sh::BPC) void k_gemm16(GemmArgs a, GemmEpi e) {
    constexpr int BM = Sh::BM, BN = Sh::BN, BK = Sh::BK, RowB = Sh::RowB, Spr = Sh::Spr;
    constexpr int TM = Sh::TM, TN = Sh::TN;
    __shared__ __attribute__((aligned(16))) uint8_t smem[Sh::Smem];
    const uint32_t sbase = lds_addr(smem);
    const int tid = threadIdx.x, l = tid & 63, n = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = w / Sh::WN, wn = w % Sh::WN;
    const int M = a.M, N0 = a.N0, N1 = a.N1, K = a.K, lda = a.lda, ldb = a.ldb;
    const int tn0 = (N0 + BN - 1) / BN, tn = tn0 + (N1 + BN - 1) / BN;
    const int tm = (M + BM - 1) / BM, ntiles = tm * tn;
    // Tiles in row-major order, XCD b % 8 taking a contiguous eighth of them (blocks of one XCD
    // share A rows in its L2).
    const int xcd = blockIdx.x & 7, per = ntiles >> 3, rem = ntiles & 7;
    const int tile = xcd * per + min(xcd, rem) + (blockIdx.x >> 3);
    const int mt = tile / tn, nt = tile % tn;
    const bool seg1 = nt >= tn0;
    const uint16_t *B = seg1 ? a.B1 : a.B0;
    const int Nseg = seg1 ? N1 : N0;
    const int nb0 = seg1 ? (nt - tn0) * BN : nt * BN;  // first row of B in this tile
    const int c0 = seg1 ? N0 + nb0 : nb0;              // first column of C
    const int m0 = mt * BM;
    const bool use_lo = Sh::LO && (Sh::AF32 || (a.Al && (!a.lo_flag || *a.lo_flag)));
    if (a.clear && blockIdx.x == 0 && tid == 0) __hip_atomic_store(a.clear, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);

    const int nkt = K / BK;
    constexpr int NS = Sh::Stages;
    if (w >= Sh::MW) {
        // DMA wave dw: instruction i fills slot (4i + dw) * 64 + l of a tile: row p / Spr,
        // physical slot p % Spr holding logical slot (p % Spr) ^ swz(row). Rows past the end of
        // A or B are clamped to the last row (their results are never stored).
        const int dw = w - Sh::MW;
        constexpr int NA = Sh::ATile / (kGemmDma * 1024), NB = Sh::BTile / (kGemmDma * 1024);
        static_assert(NA >= 1 && NB >= 1, "whole DMA instructions per tile");
        uint32_t aoff[(Sh::AF32 ? 2 : 1) * NA], boff[NB];
        if constexpr (Sh::AF32) {
#pragma unroll
            for (int i = 0; i < 2 * NA; ++i) {  // fp32 rows: twice the slots, the low three bits swizzled
                const int p = (kGemmDma * i + dw) * 64 + l, row = p / (2 * Spr), s = (p % (2 * Spr)) ^ (row & 7);
                aoff[i] = (uint32_t)(min(m0 + row, M - 1) - m0) * lda * 4 + 16 * s;
            }
        } else
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int p = (kGemmDma * i + dw) * 64 + l, row = p / Spr, s = (p % Spr) ^ Sh::swz(row);
            aoff[i] = (uint32_t)(min(m0 + row, M - 1) - m0) * lda * 2 + 16 * s;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int p = (kGemmDma * i + dw) * 64 + l, row = p / Spr, s = (p % Spr) ^ Sh::swz(row);
            boff[i] = (uint32_t)(min(nb0 + row, Nseg - 1) - nb0) * ldb * 2 + 16 * s;
        }
        const uint8_t *gah = Sh::AF32 ? (const uint8_t *)(a.Af + (size_t)m0 * lda) : (const uint8_t *)(a.Ah + (size_t)m0 * lda);
        const uint8_t *gal = use_lo && !Sh::AF32 ? (const uint8_t *)(a.Al + (size_t)m0 * lda) : gah;
        const uint8_t *gb = (const uint8_t *)(B + (size_t)nb0 * ldb);
        auto stream = [&](auto lo_tag) __attribute__((always_inline)) {
            constexpr bool kLo = decltype(lo_tag)::value;
            auto issue = [&](int kt, int stage) __attribute__((always_inline)) {
                const uint32_t dst = sbase + stage * Sh::Stage + (uint32_t)dw * 1024;
                const size_t ko = (size_t)kt * RowB;
#pragma unroll
                for (int i = 0; i < (Sh::AF32 ? 2 : 1) * NA; ++i)
                    dma_b128_s(gah + (Sh::AF32 ? 2 * ko : ko), aoff[i], dst + i * (kGemmDma * 1024));
#pragma unroll
                for (int i = 0; i < NB; ++i) dma_b128_s(gb + ko, boff[i], dst + Sh::BOff + i * (kGemmDma * 1024));
                if constexpr (kLo && !Sh::AF32) {
#pragma unroll
                    for (int i = 0; i < NA; ++i)
                        dma_b128_s(gal + ko, aoff[i], dst + Sh::ALo + i * (kGemmDma * 1024));
                }
            };
#pragma unroll
            for (int q = 0; q < NS - 1; ++q)
                if (q < nkt) issue(q, q);
            int fill = NS - 1;
            for (int kt = 0; kt < nkt; ++kt) {
                // stage kt has landed when at most min(NS - 2, nkt - 1 - kt) later stages are in flight
                wait_stages<(kLo ? 2 : 1) * NA + NB, NS - 2>(min(NS - 2, nkt - 1 - kt));
                lds_barrier();  // stage kt is in LDS; every math wave is done with stage kt - 1
                if (kt + NS - 1 < nkt) issue(kt + NS - 1, fill);
                fill = fill + 1 == NS ? 0 : fill + 1;
            }
        };
        if (Sh::AF32 || use_lo) stream(std::integral_constant<bool, Sh::LO>{});
        else stream(std::false_type{});
        lds_barrier();  // the math waves' epilogue barrier
        return;
    }
    // fragment rows 16 * tile + n (n & 7 = row & 7), logical slot 4 ks + g of k-sub ks
    int frd[BK / 32];
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) frd[ks] = n * RowB + 16 * ((4 * ks + g) ^ Sh::swz(n));

    v4f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

    auto compute = [&](auto lo_tag) __attribute__((always_inline)) {
        constexpr bool kLo = decltype(lo_tag)::value;
        int slot = 0;
        for (int kt = 0; kt < nkt; ++kt) {
            lds_barrier();  // stage kt has landed (the DMA waves waited for it)
            const uint8_t *st = smem + slot * Sh::Stage;
            slot = slot + 1 == NS ? 0 : slot + 1;
#pragma unroll
            for (int ks = 0; ks < BK / 32; ++ks) {
                const uint8_t *sa = st + wm * (TM * 16) * RowB + frd[ks];
                const uint8_t *sb = st + Sh::BOff + wn * (TN * 16) * RowB + frd[ks];
                v8bf bo[TN], ao[TM], al[kLo ? TM : 1];
#pragma unroll
                for (int j = 0; j < TN; ++j) bo[j] = *(const v8bf *)(sb + j * 16 * RowB);
                if constexpr (Sh::AF32) {
#pragma unroll
                    for (int i = 0; i < TM; ++i) {
                        const uint8_t *sf = st + (wm * TM * 16 + 16 * i + n) * 2 * RowB;
                        const v4f x0 = *(const v4f *)(sf + 16 * ((8 * ks + 2 * g) ^ (n & 7)));
                        const v4f x1 = *(const v4f *)(sf + 16 * ((8 * ks + 2 * g + 1) ^ (n & 7)));
                        split8_cvt(x0, x1, ao[i], al[kLo ? i : 0]);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < TM; ++i) ao[i] = *(const v8bf *)(sa + i * 16 * RowB);
                }
                if constexpr (kLo && !Sh::AF32) {
#pragma unroll
                    for (int i = 0; i < TM; ++i)
                        al[i] = *(const v8bf *)(sa + Sh::ALo + i * 16 * RowB);
                }
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) acc[i][j] = mfma16<F16>(ao[i], bo[j], acc[i][j]);
                if constexpr (kLo) {
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int j = 0; j < TN; ++j) acc[i][j] = mfma16<F16>(al[i], bo[j], acc[i][j]);
                }
            }
        }
    };
    if (Sh::AF32 || use_lo) compute(std::integral_constant<bool, Sh::LO>{});
    else compute(std::false_type{});
    // Epilogue. D layout: lane (g, n) of tile (i, j) holds rows 4g + r, column n. Row-major
    // outputs go through a per-wave LDS buffer (16 rows x CW = 16 TN columns per tile row i): lane
    // l then takes columns 4 (l % LR) .. + 3 of rows l / LR + RP q, so the LR lanes of a row
    // write its CW columns as one contiguous run (scattered 16-byte pieces per lane cost
    // ~10 us more per launch at these sizes), and the rope pairs (2p, 2p+1) sit in one lane.
    // The V^T part of kEpiKV wants 4 consecutive tokens per lane, which the D layout gives.
    static_assert(TN == 4 || EPI != kEpiKV, "a wave's columns of kEpiKV are all keys or all values");
    if constexpr (TN < 4 && EPI == kEpiPlain) {  // stored from the D layout, 64-byte runs
        lds_barrier();  // the DMA waves' last barrier
        float al = e.alpha;
        if (e.nan_flag && __hip_atomic_load(e.nan_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            al = __builtin_nanf("");
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int c = c0 + wn * TN * 16 + 16 * j + n;
                if (c - c0 + nb0 >= Nseg) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int t = m0 + wm * TM * 16 + 16 * i + 4 * g + r;
                    if (t < M) a.C[(size_t)t * a.ldc + c] = acc[i][j][r] * al;
                }
            }
        return;
    } else {
    const int QD = e.DN + e.DR, KH = e.DN + e.DV;
    lds_barrier();  // every wave is done with the ring
    constexpr int CW = 16 * TN, LR = CW / 4, RP = 64 / LR, EpS = CW + 4;
    float *ep = (float *)smem + w * (16 * EpS);
    const int cw = wn * CW;                      // wave's first column within the tile
    const bool vt_wave = EPI == kEpiKV && ((nb0 + cw) % KH) >= e.DN;
    const int rr = l / LR, cc = (l % LR) * 4;    // staged row (+ RP q) / first column of this lane
    const int nl0 = nb0 + cw + cc;               // segment column of v[0]
    float alpha = e.alpha;
    if (EPI == kEpiPlain && e.nan_flag && __hip_atomic_load(e.nan_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        alpha = __builtin_nanf("");
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int rbase = m0 + wm * TM * 16 + 16 * i;
        if (vt_wave) {
            const int row0 = rbase + 4 * g;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int nl = nb0 + cw + 16 * j + n;
                if (nl >= Nseg) continue;
                const int h = nl / KH, d = nl % KH - e.DN;
                const v4h hv = {(_Float16)(acc[i][j][0] * e.vscale), (_Float16)(acc[i][j][1] * e.vscale),
                                (_Float16)(acc[i][j][2] * e.vscale), (_Float16)(acc[i][j][3] * e.vscale)};
                const size_t o = ((size_t)h * e.DV + d) * e.Sp + (row0 & ~31) + vt_perm(row0 & 31);
                if (row0 + 3 < M) {
                    *(v4h *)(e.vt + o) = hv;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (row0 + r < M) e.vt[o + r] = hv[r];
                }
            }
            continue;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) ep[(4 * g + r) * EpS + 16 * j + n] = acc[i][j][r];
        v4f vq[16 / RP];
#pragma unroll
        for (int q = 0; q < 16 / RP; ++q) vq[q] = *(const v4f *)(ep + (rr + RP * q) * EpS + cc);
        if (nl0 >= Nseg) continue;
#pragma unroll
        for (int q = 0; q < 16 / RP; ++q) {
            const int t = rbase + rr + RP * q;
            if (t >= M) continue;
            if (EPI == kEpiPlain || (EPI == kEpiQ && seg1)) {
                float *dst = EPI == kEpiPlain ? a.C + (size_t)t * a.ldc + c0 + cw + cc : a.C + (size_t)t * a.ldc + nl0;
                *(v4f *)dst = EPI == kEpiPlain ? vq[q] * alpha : vq[q];
            } else if (EPI == kEpiQ) {
                store_q4(e, t, nl0, vq[q]);
            } else {  // kEpiKV, k_nope columns
                const int h = nl0 / KH, k0 = nl0 % KH;
                const size_t o = ((size_t)h * e.Sp + t) * QD + k0;
                v4h hi, lo;
                split4_f16(vq[q], hi, lo);
                *(v4h *)(e.kh + o) = hi;
                uint8_t *row = e.k8 + ((size_t)h * e.Sp + t) * 384 + k8_hi_byte(k0);
                *(uint32_t *)row = f16x4_to_bf8(hi);
                *(uint32_t *)(row + kK8Lo) = bf8_lo_s11(lo);
            }
        }
    }
    }
}

// C = A . [B0; B1]^T with N0 + N1 output columns (N1 = 0: a single weight matrix).
//
// The tile shape goes by the number of tiles the call gives: a launch takes as many rounds of its
// blocks as 256 CUs need, and a round of a shape takes about the same time whatever the number of
// its blocks, so the shape with the smallest rounds x time per round runs. Below a few hundred
// tokens a large tile leaves most CUs idle and a block's time is the latency of its k loop, which
// small tiles hide with deeper rings; above a few thousand the bytes a CU takes in per MFMA decide
// for the large ones. The times per round (gemm_pick) are of q | kv_a and kv_b launches with the lo
// part: whether x has one is known on the device only. Stand-alone launches back to back (K = 2048 for
// q | kv_a and o_proj, 512 for kv_b), tokens -> us of the chosen shape, in brackets that of the 256-row
// tiles with two passes over k that every size took before:
//   q | kv_a  250: 15.3 (50)  1181: 44 (55)  4096: 108 (134)  16000: 415, without a lo part 13.3, 35, 67, 257
//   kv_b      250: 5.6 (21)   1181: 18 (24)  4096: 41 (50)    16000: 151 (171)
//   o_proj    250: 8.1 (24)   1181: 18 (27)  4096: 34 (38)    16000: 117 (118)
// Without a lo part the choice is within a tenth of the best shape but for q alone at 2561 to 4096 tokens
// (128 x 128: 97 us with, 70 without a lo part at 4096; 256 x 256: 101 and 61). Within a call, operands
// from memory and the clock under load, a launch takes up to a quarter longer (q | kv_a at 4096: 134).
template <class Sh, int EPI, bool F16>
static hipError_t gemm_launch(hipStream_t st, const GemmArgs &a, const GemmEpi &e, int tiles) {
    hipLaunchKernelGGL((k_gemm16<Sh, EPI, F16>), dim3(tiles), dim3(Sh::Threads), 0, st, a, e);
    return hipGetLastError();
}

enum { kTile64x64 = 0, kTile128x64, kTile128x128, kTile192x128, kTile256x128, kTile256x256, kGemmTiles };

// The q (| kv_a) projection of a short prompt, from fp32 x when x is given (16-byte aligned; *clear is
// then cleared, which k_split does otherwise), else from the planes. Every tile sums the whole of k in
// one order, as the tiles of longer prompts do, so a token's Q and kv_a do not depend on how many tokens
// follow it (k split over 4 blocks, its sums added by k_kva_pack, gave 30.2 us for 37 tokens in all where
// this gives 35.3, and lost that). A block's time is the serial chain of its 64 k-subs (LDS reads, splits,
// MFMAs; stages of 128 or 256 k change nothing), so the smallest tile that still gives every tile a CU
// runs. us with weights in the caches / from memory, 32 x 32, 32 x 64, 64 x 64 (tokens x columns):
//   fp32 x, q | kv_a   37: 11.3 / 15.0  13.5 / 17.8  14.5 / 21.7   128: 19.7 / 23.2  14.3 / 20.4  15.5 / 23.9
//   planes, q alone    37:  7.7 / 14.5   9.8 / 17.5  11.0 / 22.2   160: 13.7 / 20.9  13.1 / 19.8  13.9 / 23.8
//   fp32 x, q | kv_a  160: 27.7 / 31.2  24.3 / 28.5  15.8 / 24.1
// The planes are 3 us quicker to multiply than fp32 x at 37 tokens, the k_split launch costs 2.3.
template <class P, class F>
static hipError_t gemm_q_launch(hipStream_t st, const GemmArgs &a, const GemmEpi &e) {
    const int tiles = (a.M + P::BM - 1) / P::BM * ((a.N0 + P::BN - 1) / P::BN + (a.N1 + P::BN - 1) / P::BN);
    return a.Af ? gemm_launch<F, kEpiQ, false>(st, a, e, tiles) : gemm_launch<P, kEpiQ, false>(st, a, e, tiles);
}

static hipError_t gemm_q_small(hipStream_t st, const float *x, int *clear, const uint16_t *Ah, const uint16_t *Al,
                               const int *flag, const uint16_t *B0, int N0, const uint16_t *B1, int N1, float *C, int M,
                               int K, const GemmEpi &e) {
    const GemmArgs a{Ah, Al, B0, B1 ? B1 : B0, C, flag, M, N0, N1, K, K, K, N1, x, x ? clear : nullptr};
    if (K % 64) return hipErrorInvalidValue;
    auto tiles = [&](int bm, int bn) { return (M + bm - 1) / bm * ((N0 + bn - 1) / bn + (N1 + bn - 1) / bn); };
    if (tiles(32, 32) <= 256)
        return gemm_q_launch<GemmCfg<32, 32, 64, 2, 2, true>, GemmCfg<32, 32, 64, 2, 2, true, true>>(st, a, e);
    if (tiles(32, 64) <= 256)
        return gemm_q_launch<GemmCfg<32, 64, 64, 2, 2, true>, GemmCfg<32, 64, 64, 2, 2, true, true>>(st, a, e);
    return gemm_q_launch<GemmCfg<64, 64, 64, 4, 2, true>, GemmCfg<64, 64, 64, 4, 2, true, true>>(st, a, e);
}

static int gemm_pick(int epi, int M, int N0, int N1, int *tiles) {
    static const int bm[kGemmTiles] = {64, 128, 128, 192, 256, 256}, bn[kGemmTiles] = {64, 64, 128, 128, 128, 256};
    // [epilogue]: us per round of 256 blocks (64 x 64: two blocks fit a CU, us up to 256 blocks; a
    // round of 512 takes kTwo us)
    static const float cost[3][kGemmTiles] = {{11.0f, 13.0f, 19.0f, 24.0f, 31.0f, 52.0f},
                                              {15.0f, 22.0f, 29.0f, 45.0f, 52.0f, 101.0f},
                                              {6.0f, 9.2f, 13.5f, 18.5f, 23.0f, 40.0f}};
    static const float kTwo[3] = {20.0f, 24.0f, 9.8f};
    int best = 0;
    float tbest = 0.0f;
    for (int c = 0; c < kGemmTiles; ++c) {
        const int n = (M + bm[c] - 1) / bm[c] * ((N0 + bn[c] - 1) / bn[c] + (N1 + bn[c] - 1) / bn[c]);
        const float t = c == kTile64x64 ? (n <= 256 ? cost[epi][c] : kTwo[epi] * std::max(1.0f, (n + 64) / 512.0f))
                                        : cost[epi][c] * (float)((n + 255) / 256);
        if (c == 0 || t < tbest) {
            best = c;
            tbest = t;
            *tiles = n;
        }
    }
    return best;
}

template <int EPI, bool F16 = false>
static hipError_t gemm(hipStream_t st, const uint16_t *Ah, const uint16_t *Al, const int *flag,
                       int lda, const uint16_t *B0, int N0, const uint16_t *B1, int N1, int ldb,
                       float *C, int ldc, int M, int K, const GemmEpi &e) {
    GemmArgs a{Ah, Al, B0, B1 ? B1 : B0, C, flag, M, N0, N1, K, lda, ldb, ldc, nullptr, nullptr};
    if (K % 64) return hipErrorInvalidValue;
    constexpr bool LO = !F16;  // the fp16 product has no lo operand
    if (!LO && Al) return hipErrorInvalidValue;
    int tiles = 0;
    if constexpr (EPI == kEpiPlain) {
        // half-width tiles while every one has a CU (o_proj up to 256 tokens): half the weights per
        // block; 37 tokens 8.2 -> 6.4 us, 250 tokens 8.8 -> 8.1, beyond one round slower
        tiles = (M + 63) / 64 * ((N0 + 31) / 32);
        if (N1 == 0 && tiles <= 256) return gemm_launch<GemmCfg<64, 32, 64, 4, 2, LO>, EPI, F16>(st, a, e, tiles);
    }
    switch (gemm_pick(EPI, M, N0, N1, &tiles)) {
    case kTile64x64:
        if constexpr (EPI == kEpiQ) return hipErrorInvalidValue;  // gemm_q_small's
        else return gemm_launch<GemmCfg<64, 64, 64, 4, 2, LO>, EPI, F16>(st, a, e, tiles);
    case kTile128x64: return gemm_launch<GemmCfg<128, 64, 64, 4, 1, LO>, EPI, F16>(st, a, e, tiles);
    case kTile128x128: return gemm_launch<GemmCfg<128, 128, 64, 8, 1, LO>, EPI, F16>(st, a, e, tiles);
    case kTile192x128: return gemm_launch<GemmCfg<192, 128, 64, 8, 1, LO>, EPI, F16>(st, a, e, tiles);
    case kTile256x128: return gemm_launch<GemmCfg<256, 128, 64, 8, 1, LO>, EPI, F16>(st, a, e, tiles);
    default: return gemm_launch<GemmCfg<256, 256, LO ? 32 : 64, 8, 1, LO>, EPI, F16>(st, a, e, tiles);
    }
}

// ================================================================ epilogues ============

// Per token t: latent = RMSNorm(katmp[:R]) * w (bit-exact with src/ops.c:76-83 up to the
// summation order of the double sum), stored fp32 and as hi/lo bf16; rotated k_rope
// (src/mla_prefill_streaming.c:131-138) stored fp32 [S, DR].
struct KvaEpiArgs {
    const float *y;
    const uint16_t *norm;
    const float2 *cs;
    float *latf;
    uint16_t *lath, *latl;
    float *krope;
    int *lat_flag;
    int ldy, koff, R, DR;
    float eps;
};

__global__ __launch_bounds__(256) void k_kva_epi(KvaEpiArgs a) {
    __shared__ double redd[256];
    const int t = blockIdx.x, tid = threadIdx.x, R = a.R, half = a.DR / 2;
    const float *kat = a.y + (size_t)t * a.ldy + a.koff;
    double ss = 0.0;
    for (int r = tid; r < R; r += 256) {
        const double v = (double)kat[r];
        ss += v * v;
    }
    redd[tid] = ss;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) redd[tid] += redd[tid + o];
        __syncthreads();
    }
    const float mean_sq = (float)(redd[0] / (double)R);
    const float inv = 1.0f / sqrtf(mean_sq + a.eps);
    int any = 0;
    for (int r = tid; r < R; r += 256) {
        const float v = kat[r] * inv;
        const float y = v * bf16_to_f32(a.norm[r]);
        a.latf[(size_t)t * R + r] = y;
        if (a.lath) {
            uint16_t h, l;
            split_bf16(y, h, l);
            a.lath[(size_t)t * R + r] = h;
            a.latl[(size_t)t * R + r] = l;
            any |= (l & 0x7fff) != 0;
        }
    }
    for (int i = tid; i < half; i += 256) {
        const float2 cs = a.cs[(size_t)t * half + i];
        const float ev = kat[R + 2 * i], od = kat[R + 2 * i + 1];
        const float ec = ev * cs.x, os = od * cs.y, oc = od * cs.x, es = ev * cs.y;
        a.krope[(size_t)t * a.DR + i] = ec - os;
        a.krope[(size_t)t * a.DR + half + i] = oc + es;
    }
    if (a.lat_flag && __syncthreads_or(any) && tid == 0) atomicOr(a.lat_flag, 1);
}

// MFMA route, one wave per token t: latent = RMSNorm(kv_a[t, :R]) * w (as k_kva_epi) as
// hi/lo bf16 [S, R] for the kv_b GEMM (whose lo pass always runs), and the rotated k_rope
// (src/mla_prefill_streaming.c:131-138) into the rope part of K for every head, as the fp16
// hi row and the K8 bytes (bf8 of hi and of lo x 2^11). The V^T entries of the padding keys S ..
// Sp - 1 are zeroed (their weights are exactly 0 in the flash kernel, whose mask sets their scores
// whatever Q and K hold there; rows of padding queries are not stored). Blocks past the tokens do
// that: with every token's wave also zeroing Q, K and K8 of a padding token, 37 tokens took 9.6 us.
struct KvaPackArgs {
    const float *y;  // [S, ldy] kv_a projection
    const uint16_t *norm;
    const float2 *cs;
    uint16_t *lath, *latl;
    _Float16 *kh;
    uint8_t *k8;
    _Float16 *vt;
    size_t pstride;  // np partials of y, pstride floats apart, summed in order
    int np, S, Sp, NH, ldy, R, DN, DR, DV;
    float eps;
    int *x_flag;     // the x lo flag, cleared for the next prefill (its one reader has run)
};

__global__ __launch_bounds__(256) void k_kva_pack(KvaPackArgs a) {
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
    if (blockIdx.x == 0 && threadIdx.x == 0 && a.x_flag) *a.x_flag = 0;
    const int QD = a.DN + a.DR, half = a.DR / 2, R = a.R;
    const int tblocks = (a.S + 3) / 4;
    if ((int)blockIdx.x >= tblocks) {  // padding keys of V^T: 16 rows (h, d) per wave, one key per lane
        const int r0 = 16 * (t - 4 * tblocks);
        for (int r = r0; r < min(r0 + 16, a.NH * a.DV); ++r)
            for (int k = a.S + l; k < a.Sp; k += 64) a.vt[(size_t)r * a.Sp + (k & ~31) + vt_perm(k & 31)] = 0;
        return;
    }
    if (t >= a.S) return;
    const float *kat = a.y + (size_t)t * a.ldy;
    if (R == 512 && a.DR == 64 && (a.DN & 63) == 0 && (a.ldy & 3) == 0 && (a.pstride & 3) == 0) {
        // lane l: latent columns 8l .. 8l+7 (16-byte loads and stores); the rotated RoPE key
        // goes through LDS so that each head's 128-byte fp16 hi row and its 128 K8 bytes (the
        // rope dims are k-block pair DN / 64: 4 hi slots, 4 lo slots) are written by 16 lanes of
        // 16 bytes, four heads per store instruction
        __shared__ __attribute__((aligned(16))) _Float16 rp[4][64];
        __shared__ __attribute__((aligned(16))) uint8_t k8p[4][8][16];  // [wave][part * 4 + g]
        const int w = threadIdx.x >> 6;
        float v[8];
        {
            v4f p0 = *(const v4f *)(kat + 8 * l), p1 = *(const v4f *)(kat + 8 * l + 4);
            for (int q = 1; q < a.np; ++q) {
                p0 += *(const v4f *)(kat + (size_t)q * a.pstride + 8 * l);
                p1 += *(const v4f *)(kat + (size_t)q * a.pstride + 8 * l + 4);
            }
            v[0] = p0.x; v[1] = p0.y; v[2] = p0.z; v[3] = p0.w;
            v[4] = p1.x; v[5] = p1.y; v[6] = p1.z; v[7] = p1.w;
        }
        double ss = 0.0;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += (double)v[e] * (double)v[e];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
        const float inv = 1.0f / sqrtf((float)(ss / (double)R) + a.eps);
        const v4i nw = *(const v4i *)(a.norm + 8 * l);
        uint32_t hw[4], lw[4];
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const uint32_t u = (uint32_t)nw[e >> 1];
            uint16_t h0, l0, h1, l1;
            split_bf16((v[e] * inv) * __uint_as_float(u << 16), h0, l0);
            split_bf16((v[e + 1] * inv) * __uint_as_float(u & 0xffff0000u), h1, l1);
            hw[e >> 1] = pack2(h0, h1);
            lw[e >> 1] = pack2(l0, l1);
        }
        *(v4i *)(a.lath + (size_t)t * R + 8 * l) = v4i{(int)hw[0], (int)hw[1], (int)hw[2], (int)hw[3]};
        *(v4i *)(a.latl + (size_t)t * R + 8 * l) = v4i{(int)lw[0], (int)lw[1], (int)lw[2], (int)lw[3]};
        if (l < 32) {
            const float2 cs = a.cs[(size_t)t * 32 + l];
            float ev = kat[R + 2 * l], od = kat[R + 2 * l + 1];
            for (int q = 1; q < a.np; ++q) {
                ev += kat[(size_t)q * a.pstride + R + 2 * l];
                od += kat[(size_t)q * a.pstride + R + 2 * l + 1];
            }
            const float ec = ev * cs.x, os = od * cs.y, oc = od * cs.x, es = ev * cs.y;
            _Float16 h0, l0, h1, l1;
            split_f16(ec - os, h0, l0);
            split_f16(oc + es, h1, l1);
            rp[w][l] = h0;
            rp[w][32 + l] = h1;
            // dims DN + l (k-block 2p) and DN + 32 + l (2p + 1): group (l >> 3) & 3, element l & 7
            const int g8 = (l >> 3) & 3, e = l & 7;
            k8p[w][g8][e] = (uint8_t)f16_to_bf8(h0);
            k8p[w][g8][8 + e] = (uint8_t)f16_to_bf8(h1);
            k8p[w][4 + g8][e] = (uint8_t)bf8_lo_s11(l0);
            k8p[w][4 + g8][8 + e] = (uint8_t)bf8_lo_s11(l1);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // lanes of part 0: 16 bytes of the fp16 hi row (dims DN + 8c ..); part 1: K8 slot c & 3 of
        // the hi (c < 4) or lo part
        const int part = (l >> 3) & 1, c = l & 7;
        const v4i rv = part ? *(const v4i *)k8p[w][c] : *(const v4i *)&rp[w][8 * c];
        uint8_t *dst = part ? a.k8 + (size_t)t * 384 + (c < 4 ? 0 : kK8Lo) + 16 * (4 * (a.DN >> 6) + (c & 3))
                            : (uint8_t *)(a.kh + (size_t)t * QD + a.DN + 8 * c);
        const size_t hs = part ? (size_t)a.Sp * 384 : (size_t)a.Sp * QD * sizeof(_Float16);
        for (int h = l >> 4; h < a.NH; h += 4) *(v4i *)(dst + h * hs) = rv;
        return;
    }
    auto kv = [&](int r) {
        float v = kat[r];
        for (int q = 1; q < a.np; ++q) v += kat[(size_t)q * a.pstride + r];
        return v;
    };
    double ss = 0.0;
    for (int r = l; r < R; r += 64) {
        const double v = (double)kv(r);
        ss += v * v;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
    const float mean_sq = (float)(ss / (double)R);
    const float inv = 1.0f / sqrtf(mean_sq + a.eps);
    for (int r = l; r < R; r += 64) {
        const float v = kv(r) * inv;
        const float y = v * bf16_to_f32(a.norm[r]);
        uint16_t hh, ll;
        split_bf16(y, hh, ll);
        a.lath[(size_t)t * R + r] = hh;
        a.latl[(size_t)t * R + r] = ll;
    }
    for (int i = l; i < half; i += 64) {
        const float2 cs = a.cs[(size_t)t * half + i];
        const float ev = kv(R + 2 * i), od = kv(R + 2 * i + 1);
        const float ec = ev * cs.x, os = od * cs.y, oc = od * cs.x, es = ev * cs.y;
        _Float16 h0, l0, h1, l1;
        split_f16(ec - os, h0, l0);
        split_f16(oc + es, h1, l1);
        const int b0 = k8_hi_byte(a.DN + i), b1 = k8_hi_byte(a.DN + half + i);
        const uint8_t h0b = (uint8_t)f16_to_bf8(h0), l0b = (uint8_t)bf8_lo_s11(l0);
        const uint8_t h1b = (uint8_t)f16_to_bf8(h1), l1b = (uint8_t)bf8_lo_s11(l1);
        for (int h = 0; h < a.NH; ++h) {
            const size_t o = ((size_t)h * a.Sp + t) * QD + a.DN;
            uint8_t *row = a.k8 + ((size_t)h * a.Sp + t) * 384;
            a.kh[o + i] = h0;
            row[b0] = h0b;
            row[b0 + kK8Lo] = l0b;
            a.kh[o + half + i] = h1;
            row[b1] = h1b;
            row[b1 + kK8Lo] = l1b;
        }
    }
}

// ================================================================ flash attention ======

// Causal attention for one head and 64 U queries: 8 waves, wave w taking queries 16 U (w % 4) ..
// (U 16-query tiles) and half w / 4 of every 64-key tile. QD = 192, DV = 128. Operands
// are fp16 (11 significant bits, ample range for these values): Q and K as hi + lo pairs, V and P
// rounded once.
//
// Scores are computed transposed, S^T = K Q^T (A = K from LDS, B = Q^T from registers), as
// Kh Qh (v_mfma_f32_16x16x32_f16) plus the correction Kh Ql + Kl Qh as one bf8 product over
// 384 concatenated dims (v_mfma_scale_f32_16x16x128_f8f6f4, three per 16 x 16 tile): K8 rows
// hold bf8(Kh) and bf8(Kl 2^11) per lane group, the query operand bf8(Ql 2^11) and bf8(Qh) in
// the matching byte order, and the MFMA scales the product by 2^-11. The correction terms are
// 2^-11 of the product and bf8 keeps them to 2^-3, so the score error stays near 2^-14 of
// |K||Q| even for large logits, where a single rounding of K would be amplified by the logit
// size (the Kl Ql term is below 2^-22). Lane (g, n) then holds
// S^T[key 16t + 4g + i][query n], exactly the values it must supply as the B operand of
// O^T = V^T P^T when the k-slots of a 32-key chunk are ordered (16-key tile 0: i = 0..3,
// tile 1: i = 0..3) per lane group g; V^T is stored with its keys permuted to that order
// (kv_b GEMM), so P never leaves the registers. Softmax is online with a lazy reference max
// per query: it moves only when a tile's max exceeds it by more than 8 (log2 units), so
// p <= 256 and most tiles skip the rescale.
//
// The two waves of a SIMD (w and w + 4) take the two key halves with separate running maxima and
// sums, and work half a step apart, so that one's softmax runs under the other's MFMAs: both run
// the same loop (QK of tile j, then its softmax and PV), the first passing the barrier of step j
// before QK(j), the second that of step j + 1 after it. K tiles stream through a two-slot LDS ring
// and V tiles through a three-slot one (the second half reads V one step later), filled by
// global_load_lds_dwordx4 DMA one step ahead; each half issues its share after its QK, under the
// other's MFMAs (the 64 KB take a quarter of a step to issue). The halves are merged through LDS at
// the end. The 16-byte slots of each LDS row are XOR-swizzled by the row so that the fragment reads
// are free of bank conflicts.
//
// Bound by the serial chain of a wave's step (LDS reads -> MFMAs -> softmax -> MFMAs) and the DMA
// rather than by one unit (16000 tokens: MFMA busy for about 930 us), short prompts by the prologue
// and by fetching the code once. Measured alone (us, 37 / 1181 / 4096 / 16000 tokens):
//   11.2 / 46.0 / 161 / 1944  one wave per SIMD (32 queries, all 64 keys), hand-interleaved
//   11.6 / 44.6 / 160 / 1992  two, on the key halves
//   11.1 / 41.0 / 148 / 1787  the cross-lane max taken only when it moves, bf8 by hardware
//   10.9 / 37.5 / 144 / 1763  the DMA of the two halves apart
//   11.0 / 36.5 / 139 / 1700  one loop for both, K fragments read two groups ahead (two copies of
//                             the loop left the compiler too few registers for that)
//   10.3 / 36.0 / 139 / 1687  V fragments read before the weights, one copy of the merge
//    6.2 / 24.2 / 139 / 1687  U = 1 up to kFlashSmall blocks of 128 queries
constexpr int kFK = 64;
constexpr int kFKB = kFK * 192 * 2;  // K tile (hi or lo): 64 rows x 384 B
constexpr int kFVB = 128 * kFK * 2;  // V^T tile: 128 rows x 128 B
constexpr int kFSmem = 2 * 2 * kFKB + 3 * kFVB;
constexpr int kFlashSmall = 256;     // blocks of 128 queries up to which blocks of 64 are taken
constexpr float kFLazy = 8.0f;       // log2 headroom of the lazy max
constexpr float kFNone = -1e30f;     // running max of a key half that has seen no key yet (finite:
                                     // differences of it and of itself stay numbers)

struct FlashArgs {
    const _Float16 *qh, *kh;                 // Q, K hi: [NH, Sp, 192]
    const uint8_t *ql8;                      // bf8(Q lo x 2^11): [NH, Sp, 192]
    const uint8_t *k8;                       // K8 rows: [NH, Sp, 384 bytes]
    const _Float16 *vt;                      // V^T: [NH, 128, Sp]
    _Float16 *o;                             // [S, ldo] fp16 (input of the o_proj GEMM)
    int *flag_call, *flag_sticky;            // range flags (flag_sticky may be null)
    int S, Sp, NH, ldo;
    float sl2;                               // softmax scale * log2(e)
};

// Largest |row max logit| (natural units, scale included) for which the scores' bf8
// correction keeps the attention within the 2e-3 budget with margin: measured at 256 tokens,
// row-max logits up to ~150 give 3e-4, ~500 give 6e-4, ~1450 give 1.7e-3, ~4400 give 2.3e-3.
constexpr float kFLogitMax = 512.0f;

// v_maximum3_f32: two operations that the compiler knows, so that it puts the wait states an MFMA
// result needs in front of them. A NaN score makes the maximum NaN, which raises nothing; its weight
// makes the query's sum and outputs NaN, which the range check finds.
__device__ __forceinline__ float max3(float a, float b, float c) {
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}
// Max / sum over the four lanes n, n + 16, n + 32, n + 48 (one per 16-lane row).
__device__ __forceinline__ float xrow_max(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
__device__ __forceinline__ float xrow_sum(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

template <int U>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_flash_prefill(FlashArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[kFSmem];
    const uint32_t sbase = lds_addr(smem);
    const int tid = threadIdx.x, l = tid & 63, n = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), half = w >> 2;
    // kernel arguments as locals (the lambdas below must not capture the argument block)
    const int S = a.S, Sp = a.Sp, NH = a.NH, ldo = a.ldo;
    const float sl2 = a.sl2;
    constexpr int FQ = 64 * U;  // queries of a block
    const int nqt = (S + FQ - 1) / FQ;
    // Longest tiles first; with NH % 8 == 0, block b runs on XCD b % 8 and each XCD keeps
    // the same NH / 8 heads, so the blocks streaming one head's K/V share an L2.
    int qt, h;
    if (NH % 8 == 0) {
        const int hpx = NH / 8, j = blockIdx.x >> 3;
        qt = nqt - 1 - j / hpx;
        h = (blockIdx.x & 7) + 8 * (j % hpx);
    } else {
        qt = nqt - 1 - (int)blockIdx.x / NH;
        h = (int)blockIdx.x % NH;
    }
    const int nt = U * (qt + 1);  // key tiles 0 .. nt-1 (the last U straddle the diagonal)
    const int qw = qt * FQ + 16 * U * (w & 3);
    const size_t hq = (size_t)h * Sp;

    // DMA sources. K tile: wave w fills LDS slots (3w + i) * 64 + l (16 B each) of the
    // 1536-slot tile; slot (row, s') holds logical slot s = s' ^ (row & 7) (within groups
    // of 8). V^T tile: slots (2w + i) * 64 + l of 1024; row d, slot s' holds s' ^ (d & 7).
    const uint8_t *gkh = (const uint8_t *)(a.kh + hq * 192);
    const uint8_t *gkl = a.k8 + hq * 384;
    const uint8_t *gv = (const uint8_t *)(a.vt + (size_t)h * 128 * Sp);
    uint32_t koff[3], voff[2];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int p = (3 * w + i) * 64 + l, row = p / 24, sp = p % 24;
        koff[i] = row * 384 + 16 * ((sp & ~7) | ((sp & 7) ^ (row & 7)));
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int p = (2 * w + i) * 64 + l, d = p >> 3, sp = p & 7;
        voff[i] = (uint32_t)d * Sp * 2 + 16 * (sp ^ (d & 7));
    }
    // LDS: K ring [2][hi, lo], then V ring [3]; vs: V slot of tile t
    auto issue = [&](int t, int vs) __attribute__((always_inline)) {
        const uint32_t kd = sbase + (t & 1) * 2 * kFKB + (uint32_t)(3 * w) * 1024;
        const uint32_t vd = sbase + 4 * kFKB + vs * kFVB + (uint32_t)(2 * w) * 1024;
        const size_t so = (size_t)t * kFK * 384;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            dma_b128_s(gkh + so, koff[i], kd + i * 1024);
            dma_b128_s(gkl + so, koff[i], kd + kFKB + i * 1024);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) dma_b128_s(gv + (size_t)t * 128, voff[i], vd + i * 1024);
    };
    issue(0, 0);

    // Query tile u of a wave of the second half is tile 1 - u of the first: the merge below is then
    // the same code for both (the kernel's first pass through its code is instruction fetch).
    int qu[U];  // this lane's query of tile u
#pragma unroll
    for (int u = 0; u < U; ++u) qu[u] = qw + 16 * (U == 2 ? u ^ half : 0) + n;
    // Q^T B operands: query qu[u], dims 32kb + 8g .. +7: hi as fp16 (main pass), lo as
    // its bf8(lo x 2^11) bytes (the correction operand below, written so by the q GEMM)
    v8h qa[U][6];
    uint2 qb[U][6];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const _Float16 *ph = a.qh + (hq + qu[u]) * 192 + 8 * g;
        const uint8_t *pl = a.ql8 + (hq + qu[u]) * 192 + 8 * g;
#pragma unroll
        for (int kb = 0; kb < 6; ++kb) {
            qa[u][kb] = *(const v8h *)(ph + 32 * kb);
            qb[u][kb] = *(const uint2 *)(pl + 32 * kb);
        }
    }
    // LDS fragment offsets. K (A operand): row 32 half + 16t + n, logical slot 4kb + g.
    // V^T (A operand): row 16dt + n, logical slot 4 half + g.
    int krd[6];
#pragma unroll
    for (int kb = 0; kb < 6; ++kb)
        krd[kb] = (32 * half + n) * 384 + 16 * (8 * (kb >> 1) + ((4 * (kb & 1) + g) ^ (n & 7)));
    const int vrd = n * 128 + 16 * ((4 * half + g) ^ (n & 7));
    // K8 (A operand of correction MFMA m): the same row, logical slots 8m + g and 8m + 4 + g,
    // which are the slots of kb = 2m and 2m + 1

    // correction operands: per u, 96 bytes = bf8(Ql 2^11) then bf8(Qh), each in (k-block,
    // element) order, so that byte p meets byte p of the lane group's K8 bytes (hi, then lo);
    // MFMA m takes bytes 32m .. 32m+31
    v8i q8[U][3];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        uint32_t wd[24];
#pragma unroll
        for (int kb = 0; kb < 6; ++kb)
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const v8h &q = qa[u][kb];
                const uint32_t hi = hf == 0 ? f16x4_to_bf8(__builtin_shufflevector(q, q, 0, 1, 2, 3))
                                            : f16x4_to_bf8(__builtin_shufflevector(q, q, 4, 5, 6, 7));
                wd[2 * kb + hf] = hf == 0 ? qb[u][kb].x : qb[u][kb].y;
                wd[12 + 2 * kb + hf] = hi;
            }
#pragma unroll
        for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int j = 0; j < 8; ++j) q8[u][m][j] = (int)wd[8 * m + j];
    }
    // a use of every operand here, so that the compiler's wait for their loads stands before the
    // loop: inside it, it would wait for the tile in flight as well, in every step
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int kb = 0; kb < 6; ++kb) asm volatile("" : "+v"(qa[u][kb]));
#pragma unroll
        for (int m = 0; m < 3; ++m) asm volatile("" : "+v"(q8[u][m]));
    }

    float m_run[U], l_run[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        m_run[u] = kFNone;
        l_run[u] = 0.f;
    }
    v4f acc[8][U];
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
        for (int u = 0; u < U; ++u) acc[dt][u] = v4f{0.f, 0.f, 0.f, 0.f};
    v4f sc[2][U];

    // Scores of tile j (K slot j & 1): each accumulator receives its products in the order Kh Qh
    // for kb = 0 .. 5, then the corrections m = 0 .. 2. Six groups of four independent MFMAs and six
    // of two (twice as long); each group is followed by the fragment reads of the next but one.
    auto qk = [&](int j) __attribute__((always_inline)) {
        const uint8_t *kt = smem + (j & 1) * 2 * kFKB;
        v8h kf[2][2];
        v8i k8[2];
        auto load_kh = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < 2; ++t) kf[kb & 1][t] = *(const v8h *)(kt + t * 16 * 384 + krd[kb]);
        };
        auto load_k8 = [&](int c) __attribute__((always_inline)) {  // correction c / 2 of key tile c & 1
            const uint8_t *r = kt + kFKB + (c & 1) * 16 * 384;
            const v4i x0 = *(const v4i *)(r + krd[c & ~1]), x1 = *(const v4i *)(r + krd[c | 1]);
            k8[c & 1] = __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7);
        };
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int u = 0; u < U; ++u) sc[t][u] = v4f{0.f, 0.f, 0.f, 0.f};
        load_kh(0);
        load_kh(1);
#pragma unroll
        for (int kb = 0; kb < 6; ++kb) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int u = 0; u < U; ++u) sc[t][u] = mfma_f16(kf[kb & 1][t], qa[u][kb], sc[t][u]);
            if (kb + 2 < 6) load_kh(kb + 2);
            else load_k8(kb - 4);
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u) sc[c & 1][u] = mfma_bf8_s11(k8[c & 1], q8[u][c >> 1], sc[c & 1][u]);
            if (c + 2 < 6) load_k8(c + 2);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // softmax of this wave's half of tile j and its share of O^T += V^T P^T (V slot vs)
    auto smpv = [&](int j, int vs) __attribute__((always_inline)) {
        const uint8_t *vt = smem + 4 * kFKB + vs * kFVB + vrd;
        const int k0 = j * kFK + 32 * half;
        if (k0 + 31 > qw) {  // the diagonal
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (k0 + 16 * t + 4 * g + i > qu[u]) sc[t][u][i] = -INFINITY;
        }
        // The running max moves only when a score of the tile exceeds it by more than kFLazy, which
        // each lane can tell from its own scores; the max over a query's four lanes is taken then.
        float mx[U];
        bool over = false;
#pragma unroll
        for (int u = 0; u < U; ++u)
            mx[u] = max3(max3(max3(sc[0][u][0], sc[0][u][1], sc[0][u][2]), sc[0][u][3], sc[1][u][0]),
                         max3(sc[1][u][1], sc[1][u][2], sc[1][u][3]), sc[1][u][3]) * sl2;
#pragma unroll
        for (int u = 0; u < U; ++u) over |= mx[u] > m_run[u] + kFLazy;
        if (__any(over)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float m = xrow_max(mx[u]);
                const float mnew = m > m_run[u] + kFLazy ? m : m_run[u];
                const float alpha = __builtin_amdgcn_exp2f(m_run[u] - mnew);
                m_run[u] = mnew;
                l_run[u] *= alpha;
#pragma unroll
                for (int dt = 0; dt < 8; ++dt) acc[dt][u] *= alpha;
            }
        }
        v8h vv0[4];
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) vv0[dt] = *(const v8h *)(vt + dt * 16 * 128);
        __builtin_amdgcn_sched_barrier(0);
        v8h pb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float ps = 0.f;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float p = __builtin_amdgcn_exp2f(fmaf(sc[t][u][i], sl2, -m_run[u]));
                    ps += p;
                    pb[u][4 * t + i] = (_Float16)p;
                }
            l_run[u] += ps;
        }
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
#pragma unroll
            for (int u = 0; u < U; ++u) acc[dt][u] = mfma_f16(vv0[dt & 3], pb[u], acc[dt][u]);
            if (dt < 4) vv0[dt] = *(const v8h *)(vt + (dt + 4) * 16 * 128);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // a tile whose first key of this half comes after this wave's last query adds nothing
    auto live = [&](int j) __attribute__((always_inline)) { return j * kFK + 32 * half <= qw + 16 * U - 1; };

    // Both halves run one loop, QK(j) then softmax and PV of tile j; the second passes the barrier of
    // step j + 1 between the two, the first before QK(j). Passing the barrier of step j: tile j is in
    // LDS, and every wave is done with K(j - 1) and V(j - 2).
    auto pass = [&]() __attribute__((always_inline)) {
        wait_vmcnt<0>();
        lds_barrier();
    };
    if (half) {
        pass();
        if (1 < nt) issue(1, 1);
    }
    int vs = 0;  // V slot of tile j
    for (int j = 0; j < nt; ++j) {
        const int v1 = vs == 2 ? 0 : vs + 1, v2 = v1 == 2 ? 0 : v1 + 1;
        const int ti = j + 1 + half, vi = half ? v2 : v1;  // the tile this wave issues in this step
        if (!half) pass();
        if (live(j)) qk(j);
        if (half && j + 1 < nt) pass();
        if (ti < nt) issue(ti, vi);
        if (live(j)) smpv(j, vs);
        vs = v1;
    }

    // Merge of the two key halves. U = 2: wave w gives its query tile 1 to wave w ^ 4, whose tile 0
    // that is, and finishes its own tile 0. U = 1: the second half gives, the first finishes.
    lds_barrier();  // the ring is free
    float *xw = (float *)(smem + w * 9216), *xr = (float *)(smem + (w ^ 4) * 9216);
    if (U == 2 || half) {
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) *(v4f *)(xw + 256 * dt + 4 * l) = acc[dt][U - 1];
        xw[2048 + l] = m_run[U - 1];
        xw[2112 + l] = l_run[U - 1];
    }
    lds_barrier();
    if (U == 1 && half) return;
    // range check of each query row: the reference max (log2 units, within kFLazy of the row's
    // true max) and every output value (NaN or Inf from operands beyond the fp16 range: an
    // exponent field of ones, which the addition carries into the sign bit)
    bool bad = false;
    const float m1 = xr[2048 + l], m = fmaxf(m_run[0], m1);
    const float a0 = __builtin_amdgcn_exp2f(m_run[0] - m), a1 = __builtin_amdgcn_exp2f(m1 - m);
    const float inv = 1.0f / xrow_sum(l_run[0] * a0 + xr[2112 + l] * a1);
    if (qu[0] < S) {
        uint32_t ones = 0;
        _Float16 *o = a.o + (size_t)qu[0] * ldo + (size_t)h * 128 + 4 * g;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
            const v4f s = acc[dt][0] * a0 + *(const v4f *)(xr + 256 * dt + 4 * l) * a1;
            const v4h ov = {(_Float16)(s[0] * inv), (_Float16)(s[1] * inv), (_Float16)(s[2] * inv),
                            (_Float16)(s[3] * inv)};
            const uint2 ob = __builtin_bit_cast(uint2, ov);
            ones |= ((ob.x & 0x7c007c00u) + 0x04000400u) | ((ob.y & 0x7c007c00u) + 0x04000400u);
            *(v4h *)(o + 16 * dt) = ov;
        }
        bad = (ones & 0x80008000u) != 0 || !(fabsf(m) <= kFLogitMax * 1.4426950408889634f);  // m = logit * log2(e)
    }
    // any writer stores the same value; the readers are later kernels
    if (__builtin_amdgcn_ballot_w64(bad) != 0 && l == 0) {
        __hip_atomic_store(a.flag_call, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (a.flag_sticky) __hip_atomic_store(a.flag_sticky, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
}

// ================================================================ generic route ========

// Per token: RMSNorm latent, rotated k_rope, and Q rows [S, NH, QD] fp32 (any dims).
struct GenEpiArgs {
    const float *y;
    const uint16_t *norm;
    const float2 *cs;
    float *latf, *krope, *qf;
    int ldy, NH, DN, DR, R, QO;
    float eps;
};

__global__ __launch_bounds__(256) void k_gen_epi(GenEpiArgs a) {
    const int t = blockIdx.x, tid = threadIdx.x, half = a.DR / 2, QD = a.DN + a.DR;
    const float *row = a.y + (size_t)t * a.ldy;
    for (int i = tid; i < a.NH * QD; i += 256) {
        const int h = i / QD, k = i % QD;
        const float *q = row + (size_t)h * QD;
        float v;
        if (k < a.DN) {
            v = q[k];
        } else {
            const int j = (k - a.DN) % half;
            const float2 cs = a.cs[(size_t)t * half + j];
            const float ev = q[a.DN + 2 * j], od = q[a.DN + 2 * j + 1];
            const float ec = ev * cs.x, os = od * cs.y, oc = od * cs.x, es = ev * cs.y;
            v = (k - a.DN) < half ? ec - os : oc + es;
        }
        a.qf[(size_t)t * a.NH * QD + i] = v;
    }
    (void)a.QO;
}

// Causal attention, one block per (query t, head h), any dims; scores in global scratch.
// Queries t0 .. t0 + gridDim.x - 1 (one tile of the sequence: the score scratch holds one row
// of S scores per (query of the tile, head), so its size stays linear in S).
struct GenAttnArgs {
    const float *qf, *kv, *krope;
    float *heads, *scr;
    int S, NH, DN, DR, DV, t0;
    float smscale;
};

__global__ __launch_bounds__(256) void k_gen_attn(GenAttnArgs a) {
    __shared__ float red[256];
    const int t = a.t0 + blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int QD = a.DN + a.DR, KH = a.DN + a.DV, L = t + 1;
    const float *q = a.qf + ((size_t)t * a.NH + h) * QD;
    float *sc = a.scr + ((size_t)blockIdx.x * a.NH + h) * a.S;
    for (int j = tid; j < L; j += 256) {
        const float *kj = a.kv + (size_t)j * a.NH * KH + (size_t)h * KH;
        const float *rj = a.krope + (size_t)j * a.DR;
        // the dots in double and the score as (float)dot * scale, as
        // src/mla_prefill_streaming.c:171-174
        double acc = 0.0;
        for (int k = 0; k < a.DN; ++k) acc = fma((double)q[k], (double)kj[k], acc);
        for (int k = 0; k < a.DR; ++k) acc = fma((double)q[a.DN + k], (double)rj[k], acc);
        sc[j] = (float)acc * a.smscale;
    }
    __syncthreads();
    float m = -INFINITY;
    for (int j = tid; j < L; j += 256) m = fmaxf(m, sc[j]);
    red[tid] = m;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) red[tid] = fmaxf(red[tid], red[tid + o]);
        __syncthreads();
    }
    m = red[0];
    __syncthreads();
    float sum = 0.f;
    for (int j = tid; j < L; j += 256) {
        const float e = __expf(sc[j] - m);
        sc[j] = e;
        sum += e;
    }
    red[tid] = sum;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) red[tid] += red[tid + o];
        __syncthreads();
    }
    const float inv = 1.0f / red[0];
    for (int d = tid; d < a.DV; d += 256) {
        float acc = 0.f;
        for (int j = 0; j < L; ++j) acc = fmaf(sc[j], a.kv[(size_t)j * a.NH * KH + (size_t)h * KH + a.DN + d], acc);
        a.heads[(size_t)t * a.NH * a.DV + (size_t)h * a.DV + d] = acc * inv;
    }
}

// ================================================================ driver ===============

hipError_t launch_gemv(hipStream_t st, float *Y, int ldy, const float *X, int ldx, int B,
                       const uint16_t *W0, int out0, const uint16_t *W1, int out1, int in,
                       bool accumulate);

__global__ __launch_bounds__(256) void k_bf16_to_f16(_Float16 *dst, const uint16_t *src, size_t n, float scale) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        dst[i] = (_Float16)(bf16_to_f32(src[i]) * scale);
}

// *out = max(*out, the block's largest m): one atomic per block, and at most 256 blocks in the launches
// below, since atomics on one address take about 12 ns each (k_bf16_absmax with 4096 of them 50 us, now 10,
// k_vrow_l2max with 2048 28 us, now 9, for 8 and 2 MB).
__device__ __forceinline__ void block_max_to(unsigned m, unsigned *out) {
    __shared__ unsigned wm[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) atomicMax(out, max(max(wm[0], wm[1]), max(wm[2], wm[3])));
}

// *out = max(*out, largest |src[i]| as its bf16 word), NaN words left out (n % 8 == 0 or not; src
// 16-byte aligned). The operand ranges of a prefill's weights, once per weight upload: the host took
// 2.6 ms a layer for them (8 MB of o_proj, 2 MB of kv_b), which was most of a first prefill's 2.9 ms.
__global__ __launch_bounds__(256) void k_bf16_absmax(const uint16_t *src, size_t n, unsigned *out) {
    unsigned m = 0;
    auto take = [&](unsigned v) __attribute__((always_inline)) {
        v &= 0x7fffu;
        m = max(m, v <= 0x7f80u ? v : 0u);
    };
    const size_t n8 = n / 8;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (size_t)gridDim.x * 256) {
        const v4i x = *(const v4i *)(src + 8 * i);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            take((unsigned)x[k]);
            take((unsigned)x[k] >> 16);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 7)) take(src[8 * n8 + threadIdx.x]);
    block_max_to(m, out);
}

// *out = max(*out, largest L2 norm of kv_b's V rows as an fp32 word), NaN left out: one wave per row,
// double sums.
__global__ __launch_bounds__(256) void k_vrow_l2max(const uint16_t *kvb, int NH, int DN, int DV, int R, unsigned *out) {
    const int l = threadIdx.x & 63;
    unsigned m = 0;
    for (int r = blockIdx.x * 4 + (threadIdx.x >> 6); r < NH * DV; r += gridDim.x * 4) {
        const uint16_t *row = kvb + ((size_t)(r / DV) * (DN + DV) + DN + r % DV) * R;
        double ss = 0.0;
        for (int k = l; k < R; k += 64) {
            const double v = (double)bf16_to_f32(row[k]);
            ss += v * v;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
        const float f = (float)sqrt(ss);
        if (f == f) m = max(m, __float_as_uint(f));
    }
    block_max_to(m, out);
}

hipError_t launch_bf16_absmax(hipStream_t st, const uint16_t *src, size_t n, unsigned *out) {
    if (((uintptr_t)src % 16) != 0 || n == 0) return hipErrorInvalidValue;
    const int blocks = (int)std::min<size_t>(256, (n + 2047) / 2048);
    hipLaunchKernelGGL(k_bf16_absmax, dim3(blocks), dim3(256), 0, st, src, n, out);
    return hipGetLastError();
}

hipError_t launch_vrow_l2max(hipStream_t st, const uint16_t *kvb, const Dims &d, unsigned *out) {
    hipLaunchKernelGGL(k_vrow_l2max, dim3(std::min(256, (d.NH * d.DV + 3) / 4)), dim3(256), 0, st, kvb, d.NH, d.DN, d.DV, d.R, out);
    return hipGetLastError();
}

hipError_t launch_split(hipStream_t st, const float *src, int ld_src, uint16_t *hi, uint16_t *lo,
                        int ld_dst, int rows, int cols) {
    if (rows < 1 || cols < 8 || cols % 8 || ld_src % 4 || ld_dst % 8 || ld_src < cols || ld_dst < cols ||
        ((uintptr_t)src % 16) || ((uintptr_t)hi % 16) || ((uintptr_t)lo % 16))
        return hipErrorInvalidValue;
    const int blocks = std::min(2048, rows);  // k_split loops over rows by block
    hipLaunchKernelGGL(k_split, dim3(blocks), dim3(256), 0, st, src, ld_src, hi, lo, ld_dst, rows, cols,
                       nullptr);
    return hipGetLastError();
}

hipError_t launch_bf16_to_f16(hipStream_t st, _Float16 *dst, const uint16_t *src, size_t n, float scale) {
    const int blocks = (int)std::min<size_t>(4096, (n + 255) / 256);
    hipLaunchKernelGGL(k_bf16_to_f16, dim3(blocks), dim3(256), 0, st, dst, src, n, scale);
    return hipGetLastError();
}

bool prefill_mfma_shape(const Dims &d) {
    return d.H % 64 == 0 && d.R % 64 == 0 && d.QD == 192 && d.DV == 128 && d.HO % 64 == 0 &&
           d.DN % 8 == 0;
}

bool prefill_kva_exact(const Dims &d) { return prefill_mfma_shape(d) && gemv_ksplit_ok(d.H, d.H); }

// Queries per launch of the generic route's attention: the score scratch (queries x NH x S
// fp32) stays within 64 MiB, or one query's NH x S when that alone is larger.
static int gen_query_tile(const Dims &d, int S) {
    const size_t per_query = (size_t)d.NH * (size_t)S;
    const size_t cap = (size_t)16 << 20;  // floats
    return (int)std::max<size_t>(1, std::min<size_t>((size_t)S, cap / per_query));
}

size_t prefill_bytes(const Dims &d, int S, bool generic) {
    const size_t Sp = (size_t)(S + 127) / 128 * 128;
    size_t b = 0;
    auto add = [&](size_t n) { b += (n + 255) / 256 * 256 + 256; };
    if (prefill_mfma_shape(d) && !generic) {
        add(4 * 8);                              // flags
        add(2 * (size_t)S * d.H);                // x hi
        add(2 * (size_t)S * d.H);                // x lo
        add(4 * (size_t)S * d.KVO * (prefill_kva_exact(d) ? kGemvKs : 1));  // kv_a projection
        add(2 * (size_t)S * d.R);                // latent hi
        add(2 * (size_t)S * d.R);                // latent lo
        add(2 * (size_t)d.NH * Sp * d.QD);       // q hi (fp16)
        add(2 * (size_t)d.NH * Sp * d.QD);       // q lo
        add(2 * (size_t)d.NH * Sp * d.QD);       // k hi
        add(2 * (size_t)d.NH * Sp * d.QD);       // k lo
        add(2 * (size_t)d.NH * d.DV * Sp);       // v^T
        add(2 * (size_t)S * d.HO);               // heads (fp16)
    } else {
        add(4 * (size_t)S * (d.QO + d.KVO));
        add(4 * (size_t)S * d.R);
        add(4 * (size_t)S * d.DR);
        add(4 * (size_t)S * d.NH * d.QD);
        add(4 * (size_t)S * d.KVB);
        add(4 * (size_t)S * d.HO);
        add(4 * (size_t)gen_query_tile(d, S) * d.NH * S);
    }
    return b;
}

hipError_t launch_prefill_all(hipStream_t st, const Dims &d, int S, float eps, const float *x,
                              float *out, const uint16_t *wq, const uint16_t *wkva,
                              const uint16_t *wnorm, const uint16_t *wkvb, const uint16_t *wo,
                              const _Float16 *wo16, const float2 *cs, void *ws, PrefillKva *kva,
                              const PrefillRange *range) {
    const int Sp = (S + 127) / 128 * 128;
    if (kva) *kva = PrefillKva{nullptr, 0, 0, 0};
    char *base = (char *)ws;
    size_t off = 0;
    auto take = [&](size_t n) {
        off = (off + 255) / 256 * 256;
        void *p = base + off;
        off += n + 256;
        return p;
    };
    const float smscale = 1.0f / sqrtf((float)d.QD);
    const int ldy = d.QO + d.KVO;
    hipError_t e;
    if (prefill_mfma_shape(d) && !(range && range->generic)) {
        int *flags = (int *)take(4 * 8);
        uint16_t *xh = (uint16_t *)take(2 * (size_t)S * d.H);
        uint16_t *xl = (uint16_t *)take(2 * (size_t)S * d.H);
        const bool exact = kva && prefill_kva_exact(d);
        const int np = exact ? kGemvKs : 1;
        const int qn1 = exact ? 0 : d.KVO;
        float *ykva = (float *)take(4 * (size_t)S * d.KVO * np);
        uint16_t *lath = (uint16_t *)take(2 * (size_t)S * d.R);
        uint16_t *latl = (uint16_t *)take(2 * (size_t)S * d.R);
        _Float16 *qh = (_Float16 *)take(2 * (size_t)d.NH * Sp * d.QD);
        uint8_t *ql8 = (uint8_t *)take((size_t)d.NH * Sp * d.QD);
        _Float16 *kh = (_Float16 *)take(2 * (size_t)d.NH * Sp * d.QD);
        uint8_t *k8 = (uint8_t *)take((size_t)d.NH * Sp * 384);
        _Float16 *vt = (_Float16 *)take(2 * (size_t)d.NH * d.DV * Sp);
        _Float16 *heads = (_Float16 *)take(2 * (size_t)S * d.HO);
        GemmEpi ep{qh, kh, ql8, k8, vt, cs, Sp, d.DN, d.DR, d.DV};
        const float vscale = range ? range->vscale : 1.0f, oscale = range ? range->oscale : 1.0f;
        // flags[0] (any x lo word non-zero) is raised by k_split and cleared by k_kva_pack after
        // the q GEMM has read it, so no launch clears it first. A value left raised (a call
        // that failed in between, or the buffer reused by another call) only costs the GEMM's lo
        // pass over an exact plane: the flag is never clear while a lo word is non-zero.
        // A short prompt's projection takes x as it is (gemm_q_small) and needs no planes (with a state
        // fill, launch_kva_tok needs them all the same: reading fp32 x there cost more than the launch).
        int qtiles = 0;
        const bool small = gemm_pick(kEpiQ, S, d.QO, qn1, &qtiles) == kTile64x64;
        const bool direct = small && !exact && (uintptr_t)x % 16 == 0;
        if (!direct) {
            const int split_blocks = std::min(2048, S);
            hipLaunchKernelGGL(k_split, dim3(split_blocks), dim3(256), 0, st, x, d.H, xh, xl, d.H, S, d.H, flags + 0);
            if ((e = hipGetLastError()) != hipSuccess) return e;
        }
        // q (-> Q hi/lo, rotated) | kv_a (-> ykva). When the caller fills a state from this
        // kv_a, it is computed with the decode's k-split arithmetic (launch_kva_tok) so those
        // rows equal the rows a decode appends; otherwise it rides along in the q GEMM.
        if (small)
            e = gemm_q_small(st, direct ? x : nullptr, flags + 1, xh, xl, flags + 0, wq, d.QO, exact ? nullptr : wkva, qn1,
                             ykva, S, d.H, ep);
        else if (exact) e = gemm<kEpiQ>(st, xh, xl, flags + 0, d.H, wq, d.QO, nullptr, 0, d.H, nullptr, 0, S, d.H, ep);
        else e = gemm<kEpiQ>(st, xh, xl, flags + 0, d.H, wq, d.QO, wkva, d.KVO, d.H, ykva, d.KVO, S, d.H, ep);
        if (e != hipSuccess) return e;
        if (exact) {
            if ((e = launch_kva_tok(st, ykva, (size_t)S * d.KVO, d.KVO, xh, xl, S, wkva, d.KVO, d.H)) !=
                hipSuccess)
                return e;
            if (kva) *kva = PrefillKva{ykva, d.KVO, np, (size_t)S * d.KVO};
        }
        const int vpad = Sp > S ? (d.NH * d.DV + 63) / 64 : 0;
        KvaPackArgs ka{ykva, wnorm, cs, lath, latl, kh, k8, vt, (size_t)S * d.KVO, np,
                       S, Sp, d.NH, d.KVO, d.R, d.DN, d.DR, d.DV, eps, flags + 0};
        hipLaunchKernelGGL(k_kva_pack, dim3((S + 3) / 4 + vpad), dim3(256), 0, st, ka);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        // kv_b (-> K nope part as fp16 hi + K8, V^T scaled by vscale)
        ep.vscale = vscale;
        if ((e = gemm<kEpiKV>(st, lath, latl, nullptr, d.R, wkvb, d.KVB, nullptr, 0, d.R, nullptr, 0, S, d.R,
                              ep)) != hipSuccess)
            return e;
        FlashArgs fa{qh, kh, ql8, k8, vt, heads, flags + 1, range ? range->sticky : nullptr, S, Sp, d.NH, d.HO,
                     smscale * 1.4426950408889634f};
        // 64 queries per block while 128 would leave CUs without one: a launch then lasts as long as
        // its last query tile's key tiles, which U = 1 takes in less time each. 64 / 128 queries, alone
        // (us): 6.2 / 10.2 at 37 tokens, 9.2 / 14.0 at 250, 24.2 / 34.8 at 1181, 47.6 / 53.2 at 2048,
        // 81.2 / 64.0 at 2500 (320 blocks of 128).
        const int nq2 = (S + 127) / 128 * d.NH;
        if (nq2 <= kFlashSmall) hipLaunchKernelGGL(k_flash_prefill<1>, dim3((S + 63) / 64 * d.NH), dim3(512), 0, st, fa);
        else hipLaunchKernelGGL(k_flash_prefill<2>, dim3(nq2), dim3(512), 0, st, fa);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        // out = heads . o_proj^T in fp16 (heads rounded once, o_proj converted exactly), the
        // two scales undone (or NaN when the range flag of this call is up)
        if (!wo16) return hipErrorInvalidValue;
        ep.vscale = 1.0f;
        ep.alpha = 1.0f / (vscale * oscale);
        ep.nan_flag = flags + 1;
        return gemm<kEpiPlain, true>(st, (const uint16_t *)heads, nullptr, nullptr, d.HO, (const uint16_t *)wo16, d.H,
                                     nullptr, 0, d.HO, out, d.H, S, d.HO, ep);
    }
    float *y = (float *)take(4 * (size_t)S * ldy);
    float *latf = (float *)take(4 * (size_t)S * d.R);
    float *krope = (float *)take(4 * (size_t)S * d.DR);
    float *qf = (float *)take(4 * (size_t)S * d.NH * d.QD);
    float *kv = (float *)take(4 * (size_t)S * d.KVB);
    float *heads = (float *)take(4 * (size_t)S * d.HO);
    const int tq = gen_query_tile(d, S);
    float *scr = (float *)take(4 * (size_t)tq * d.NH * S);
    if ((e = launch_gemv(st, y, ldy, x, d.H, S, wq, d.QO, wkva, d.KVO, d.H, false)) != hipSuccess) return e;
    KvaEpiArgs ea{y, wnorm, cs, latf, nullptr, nullptr, krope, nullptr, ldy, d.QO, d.R, d.DR, eps};
    hipLaunchKernelGGL(k_kva_epi, dim3(S), dim3(256), 0, st, ea);
    GenEpiArgs ga{y, wnorm, cs, latf, krope, qf, ldy, d.NH, d.DN, d.DR, d.R, d.QO, eps};
    hipLaunchKernelGGL(k_gen_epi, dim3(S), dim3(256), 0, st, ga);
    if ((e = launch_gemv(st, kv, d.KVB, latf, d.R, S, wkvb, d.KVB, nullptr, 0, d.R, false)) != hipSuccess)
        return e;
    for (int t0 = 0; t0 < S; t0 += tq) {
        GenAttnArgs aa{qf, kv, krope, heads, scr, S, d.NH, d.DN, d.DR, d.DV, t0, smscale};
        hipLaunchKernelGGL(k_gen_attn, dim3(std::min(tq, S - t0), d.NH), dim3(256), 0, st, aa);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    return launch_gemv(st, out, d.H, heads, d.HO, S, wo, d.H, nullptr, 0, d.HO, false);
}

}  // namespace kvl
