// HIP kernels of the MLA decode path for MI355X (gfx950, wave64).
//
// Per decode step and launch group of up to 64 sequences:
//   gemv      q_proj | kv_a_proj projections (bf16 MFMA, x split hi/lo)
//   append    RMSNorm -> quantise (Q8) / store (FP32) -> RoPE of the key, one history row
//   qprep     absorbed query q_lat = W_UK^T q_nope and RoPE(q_rope) per head
//   attention split-K over the history, all 16 heads reuse each row read once from HBM
//   combine   merge split partials (online-softmax algebra) and apply W_UV per head
//   gemv      o_proj (optionally accumulated onto the input: residual)
// The arithmetic contract follows src/mla_compressed_q8_state.c:161-255 and
// src/mla_compressed_state.c:86-161 of the reference; the history rows produced by
// `append` are bit-exact with src/mla_compressed_q8_state.c:34-55,111-127 given the same
// kv_a output.
#include "mla_device.h"
#include "mla_internal.h"

#include <math.h>

#include <algorithm>

#include <type_traits>

namespace kvl {

// ================================================================ GEMV =================

struct GemvArgs {
    float *Y;
    const float *X;
    const uint16_t *W0;
    const uint16_t *W1;
    int ldy, ldx, B, out0, out1, in, acc;
};

constexpr int kGvKb = 8;  // k-blocks of 32 per wave and pass (at most)

// 16 output rows per block (one 16-row MFMA tile); wave w of WAVES owns the k range
// [w*in/WAVES, (w+1)*in/WAVES). Many small blocks keep every CU busy and many loads in
// flight (the kernel is latency-bound at decode batch sizes). The weight rows are the MFMA
// A operand (exact bf16), the batch of activations the B operand as a hi/lo bf16 pair, so
// every product is exact and the accumulation is fp32. Up to 16 sequences per block column
// (blockIdx.y). Requires in % (32 * WAVES) == 0 and 16-byte aligned rows.
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_gemv_mfma(GemvArgs a) {
    __shared__ v4f red[WAVES][64];
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
    const int out = a.out0 + a.out1;
    const int row = blockIdx.x * 16 + n;
    const uint16_t *wrow = row < a.out0 ? a.W0 + (size_t)row * a.in
                           : row < out  ? a.W1 + (size_t)(row - a.out0) * a.in
                                        : nullptr;
    const int b = blockIdx.y * 16 + n;
    const float *xrow = b < a.B ? a.X + (size_t)b * a.ldx : nullptr;
    const int kw = a.in / WAVES;
    const int kbeg = w * kw;
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < kw; k0 += 32 * kGvKb) {
        const int nkb = min(kGvKb, (kw - k0) >> 5);
        v4i wa[kGvKb];
        v4f xa[kGvKb], xb[kGvKb];
#pragma unroll
        for (int kb = 0; kb < kGvKb; ++kb) {
            if (kb < nkb) {
                const int k = kbeg + k0 + kb * 32 + g * 8;
                wa[kb] = wrow ? *(const v4i *)(wrow + k) : v4i{0, 0, 0, 0};
                xa[kb] = xrow ? *(const v4f *)(xrow + k) : v4f{0.f, 0.f, 0.f, 0.f};
                xb[kb] = xrow ? *(const v4f *)(xrow + k + 4) : v4f{0.f, 0.f, 0.f, 0.f};
            }
        }
#pragma unroll
        for (int kb = 0; kb < kGvKb; ++kb) {
            if (kb < nkb) {
                v8bf hi, lo;
                split8(xa[kb], xb[kb], hi, lo);
                const v8bf wv = __builtin_bit_cast(v8bf, wa[kb]);
                acc = mfma_bf16(wv, hi, acc);
                acc = mfma_bf16(wv, lo, acc);
            }
        }
    }
    red[w][l] = acc;
    __syncthreads();
    if (w == 0 && b < a.B) {
        v4f s = red[0][l];
#pragma unroll
        for (int q = 1; q < WAVES; ++q) s += red[q][l];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = blockIdx.x * 16 + 4 * g + i;
            if (r < out) {
                float *yp = a.Y + (size_t)b * a.ldy + r;
                *yp = a.acc ? *yp + s[i] : s[i];
            }
        }
    }
}

// Any shape: one wave per output row, lanes stride the input, all sequences of the group.
__global__ __launch_bounds__(256) void k_gemv_generic(GemvArgs a) {
    const int out = a.out0 + a.out1;
    const int row = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int l = threadIdx.x & 63;
    if (row >= out) return;  // whole waves leave together
    const uint16_t *wrow =
        row < a.out0 ? a.W0 + (size_t)row * a.in : a.W1 + (size_t)(row - a.out0) * a.in;
    for (int b = 0; b < a.B; ++b) {
        const float *x = a.X + (size_t)b * a.ldx;
        float s = 0.f;
        for (int i = l; i < a.in; i += 64) s = fmaf(bf16_to_f32(wrow[i]), x[i], s);
        s = wave_sum(s);
        if (l == 0) {
            float *yp = a.Y + (size_t)b * a.ldy + row;
            *yp = a.acc ? *yp + s : s;
        }
    }
}

// ---- decode projections -----------------------------------------------------------------
// Both kernels below feed the activations to the MFMA as 16 columns = bf16 hi (columns 0-7)
// and bf16 lo (columns 8-15) of 8 sequences: one MFMA per row tile and k-block carries both
// halves (the products of bf16 operands are exact in fp32), and the two columns of a sequence
// are added at the end (lanes l and l ^ 8). NG groups of 8 sequences per block, blockIdx.z
// selects the 16-sequence slice; each sequence's result is the same whatever the batch.
struct GemvSplitArgs {
    float *Y;            // k-split: partial q at Y + q * pstride; pre-split: the output
    const float *X;      // k-split: fp32 activations [B, ldx]
    const uint16_t *XS;  // pre-split: bf16 planes [2][B][in], plane 0 = hi, plane 1 = lo
    const uint16_t *W0;
    const uint16_t *W1;
    size_t pstride;
    int ldy, ldx, B, out0, out1, in, acc;
};

// Y + kq * pstride [b, o] = sum over k in [kq in/kGemvKs, (kq+1) in/kGemvKs) of W[o, k] X[b, k].
// Block: 64 output rows (4 MFMA row tiles) x one k quarter; 16 waves, each KPW 32-wide
// k-blocks for all four tiles, so every activation value a wave converts serves four MFMAs.
// Splitting k keeps the weight bytes per block at 64 KB while each block reads only a quarter
// of the activations (a 16-row block over the full k range would read all of them). The
// consumer adds the kGemvKs partials in kq order. The block takes the 16-token groups
// 16 blockIdx.z, + 16 gridDim.z, ... in turn with its weights held in registers, so a batch of
// many tokens reads each weight once. Requires in = kGemvKs * 16 * 32 * KPW.
// XCD-aware placement (kGemvKs = 4, workgroup i on XCD i % 8): the blocks of k quarter kq run
// on XCDs 2 kq and 2 kq + 1, so each XCD's L2 takes in one quarter of the activations (a
// quarter of the bytes a host-memory x crosses the bus with; the host-API decode reads x there).
// Block i: kq = (i % 8) / 2, row block 2 (i / 8) + i % 2; blocks past the last row block exit.
static_assert(kGemvKs == 4, "two XCDs per k quarter");
template <int NG, int KPW>
__global__ __launch_bounds__(1024) void k_gemv_ksplit(const float *X, const uint16_t *W0, const uint16_t *W1, size_t pstride,
                                                      int ldy, int ldx, int B, int out0, int out1, int in, float *Y,
                                                      unsigned *zf, int nz) {
    // scalar arguments: the first 14 dwords (everything but Y, which only the stores use) are
    // preloaded into SGPRs at wave start (no argument round trip)
    const GemvSplitArgs a{Y, X, nullptr, W0, W1, pstride, ldy, ldx, B, out0, out1, in, 0};
    __shared__ v4f red[16][4 * NG][64];
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
    const int xcd = blockIdx.x & 7, rb = 2 * (blockIdx.x >> 3) + (xcd & 1);
    const int out = a.out0 + a.out1, kq = xcd >> 1, row0 = rb * 64, part = n >> 3;
    // block 0 (row block 0 of k quarter 0, never empty) clears the next launch's flags (the first
    // 8 bytes of each line: the combine counters are 64 bits)
    if (blockIdx.x == 0 && zf != nullptr && tid < nz) *(uint2 *)(zf + (size_t)tid * kFqFlagStride) = uint2{0u, 0u};
    if (row0 >= out) return;  // the whole block
    const uint16_t *wr[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int row = min(row0 + 16 * t + n, out - 1);  // rows past the end are never stored
        wr[t] = row < a.out0 ? a.W0 + (size_t)row * a.in : a.W1 + (size_t)(row - a.out0) * a.in;
    }
    const int kbase = kq * (16 * 32 * KPW) + w * (32 * KPW) + g * 8;
    // the weights are read once per call: non-temporal loads keep them out of the caches
    v4i wa[KPW][4];
#pragma unroll
    for (int kb = 0; kb < KPW; ++kb)
#pragma unroll
        for (int t = 0; t < 4; ++t) wa[kb][t] = __builtin_nontemporal_load((const v4i *)(wr[t] + kbase + 32 * kb));
    // the activations of token group bz (issued one group ahead: their loads overlap the
    // reduction of the previous group)
    v4f xa[KPW][NG], xb[KPW][NG];
    auto load_x = [&](int bz) __attribute__((always_inline)) {
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
            const float *xr = a.X + (size_t)min(bz + 8 * gi + (n & 7), a.B - 1) * a.ldx;
#pragma unroll
            for (int kb = 0; kb < KPW; ++kb) {
                const int k = kbase + 32 * kb;
                xa[kb][gi] = *(const v4f *)(xr + k);
                xb[kb][gi] = *(const v4f *)(xr + k + 4);
            }
        }
    };
    load_x(16 * blockIdx.z);
    for (int bz = 16 * blockIdx.z; bz < a.B; bz += 16 * gridDim.z) {
        v4f acc[4][NG];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) acc[t][gi] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < KPW; ++kb)
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
                const v8bf xv = split8_part(xa[kb][gi], xb[kb][gi], part);
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[t][gi] = mfma_bf16(__builtin_bit_cast(v8bf, wa[kb][t]), xv, acc[t][gi]);
            }
        if (bz + 16 * gridDim.z < a.B) load_x(bz + 16 * gridDim.z);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) red[w][t * NG + gi][l] = acc[t][gi];
        __syncthreads();
        if (w < 4) {
            // wave t sums row tile t over the 16 waves in order
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
                v4f s = red[0][w * NG + gi][l];
#pragma unroll
                for (int q = 1; q < 16; ++q) s += red[q][w * NG + gi][l];
#pragma unroll
                for (int i = 0; i < 4; ++i) s[i] += dpp_f32<0x128>(s[i]);  // row_ror:8 = lane ^ 8
                const int b = bz + 8 * gi + n;
                if (n < 8 && b < a.B) {
                    float *y = a.Y + (size_t)kq * a.pstride + (size_t)b * a.ldy;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = row0 + 16 * w + 4 * g + i;
                        if (r < out) y[r] = s[i];
                    }
                }
            }
        }
        __syncthreads();  // red is rewritten by the next group
    }
}

// Y[b, o] (+)= sum_k W[o, k] (hi + lo)[b, k] with the activations already split into bf16
// planes by their producer: RB (16 or 8) output rows per block, NW waves splitting k, one
// 16-byte activation load and one MFMA per k-block and sequence group; the 16-token groups are
// taken in turn with the weights held in registers. With RB = 8, MFMA rows 8-15 repeat rows
// 0-7 and are not stored: a block then takes in 32 KB of weights instead of 64 KB beside the
// 64 KB of activations every block reads, and the grid covers twice the CUs (o_proj at batch 8:
// 6.9 -> 6.5 us). Each output is the same sum in the same order for either RB and NG. With
// in = 2048, four waves of 16 k-blocks each (the same loads in flight per block, a quarter of
// the waves to launch) measured 6.16 -> 5.89 us per launch in the batch-8 decode stack.
// Requires in = NW * 32 * KPW.
template <int NG, int KPW, int RB = 16, int NW = 16>
__global__ __launch_bounds__(64 * NW) void k_gemv_xs(float *Y, const uint16_t *XS, const uint16_t *W0, int ldy, int B,
                                                  int nout, int in, int acc, unsigned *zf, int nz) {
    // scalar arguments: preloaded into SGPRs at wave start (no argument round trip)
    const GemvSplitArgs a{Y, nullptr, XS, W0, nullptr, 0, ldy, 0, B, nout, 0, in, acc};
    static_assert(RB == 16 || RB == 8, "rows per block");
    __shared__ v4f red[NW][NG][64];
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
    // block 0 clears the flags of the fused attention launch before it (the first 8 bytes of
    // each line), for the next fused launch
    if (blockIdx.x == 0 && blockIdx.z == 0 && zf != nullptr)
        for (int k = tid; k < nz; k += 64 * NW) *(uint2 *)(zf + (size_t)k * kFqFlagStride) = uint2{0u, 0u};
    const int out = a.out0, part = n >> 3;
    const uint16_t *wrow = a.W0 + (size_t)min((int)blockIdx.x * RB + (n % RB), out - 1) * a.in;
    const int kbase = w * (32 * KPW) + g * 8;
    v4i wa[KPW];
#pragma unroll
    for (int kb = 0; kb < KPW; ++kb) wa[kb] = __builtin_nontemporal_load((const v4i *)(wrow + kbase + 32 * kb));
    v4i xv[KPW][NG];  // activations of a token group, loaded one group ahead
    auto load_x = [&](int bz) __attribute__((always_inline)) {
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) {
            const uint16_t *xr = a.XS + ((size_t)part * a.B + min(bz + 8 * gi + (n & 7), a.B - 1)) * a.in;
#pragma unroll
            for (int kb = 0; kb < KPW; ++kb) xv[kb][gi] = *(const v4i *)(xr + kbase + 32 * kb);
        }
    };
    load_x(16 * blockIdx.z);
    for (int bz = 16 * blockIdx.z; bz < a.B; bz += 16 * gridDim.z) {
        // the residual values this lane of wave 0 adds to, requested before the MFMAs and the
        // reduction so that their latency is not added at the end
        float yres[NG][4];
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int b = bz + 8 * gi + n, r = blockIdx.x * RB + 4 * g + i;
                yres[gi][i] = w == 0 && a.acc && n < 8 && 4 * g < RB && b < a.B && r < out ? a.Y[(size_t)b * a.ldy + r] : 0.f;
            }
        v4f acc[NG];
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) acc[gi] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < KPW; ++kb)
#pragma unroll
            for (int gi = 0; gi < NG; ++gi)
                acc[gi] = mfma_bf16(__builtin_bit_cast(v8bf, wa[kb]), __builtin_bit_cast(v8bf, xv[kb][gi]), acc[gi]);
        if (bz + 16 * gridDim.z < a.B) load_x(bz + 16 * gridDim.z);
#pragma unroll
        for (int gi = 0; gi < NG; ++gi) red[w][gi][l] = acc[gi];
        __syncthreads();
        if (w == 0) {
#pragma unroll
            for (int gi = 0; gi < NG; ++gi) {
                v4f s = red[0][gi][l];
#pragma unroll
                for (int q = 1; q < NW; ++q) s += red[q][gi][l];
#pragma unroll
                for (int i = 0; i < 4; ++i) s[i] += dpp_f32<0x128>(s[i]);
                const int b = bz + 8 * gi + n;
                if (n < 8 && 4 * g < RB && b < a.B) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int r = blockIdx.x * RB + 4 * g + i;
                        if (r < out) a.Y[(size_t)b * a.ldy + r] = a.acc ? yres[gi][i] + s[i] : s[i];
                    }
                }
            }
        }
        __syncthreads();  // red is rewritten by the next group
    }
}

bool gemv_ksplit_ok(int in, int ldx) { return (in == 2048 || in == 4096) && ldx % 4 == 0; }

hipError_t launch_gemv_ksplit(hipStream_t st, float *Y, size_t pstride, int ldy, const float *X,
                              int ldx, int B, const uint16_t *W0, int out0, const uint16_t *W1,
                              int out1, int in, unsigned *zero_flags, int nzero) {
    if (!gemv_ksplit_ok(in, ldx) || B < 1 || ((uintptr_t)X % 16) != 0 || ((uintptr_t)W0 % 16) != 0 ||
        (W1 && ((uintptr_t)W1 % 16) != 0) || out0 + out1 <= 0 || (B + 15) / 16 > 65535 || nzero < 0 ||
        nzero > 1024 || (nzero > 0 && zero_flags == nullptr))
        return hipErrorInvalidValue;
    // 8 blocks per pair of 64-row blocks: row blocks 2m, 2m + 1 for the four k quarters
    const int nrb = (out0 + out1 + 63) / 64;
    const dim3 grid(8 * ((nrb + 1) / 2), 1, 1);  // the block loops over the token groups
    const bool two = B > 8;
    if (in == 2048) {
        if (two) hipLaunchKernelGGL((k_gemv_ksplit<2, 1>), grid, dim3(1024), 0, st, X, W0, W1, pstride, ldy, ldx, B, out0, out1, in, Y, zero_flags, nzero);
        else hipLaunchKernelGGL((k_gemv_ksplit<1, 1>), grid, dim3(1024), 0, st, X, W0, W1, pstride, ldy, ldx, B, out0, out1, in, Y, zero_flags, nzero);
    } else {
        if (two) hipLaunchKernelGGL((k_gemv_ksplit<2, 2>), grid, dim3(1024), 0, st, X, W0, W1, pstride, ldy, ldx, B, out0, out1, in, Y, zero_flags, nzero);
        else hipLaunchKernelGGL((k_gemv_ksplit<1, 2>), grid, dim3(1024), 0, st, X, W0, W1, pstride, ldy, ldx, B, out0, out1, in, Y, zero_flags, nzero);
    }
    return hipGetLastError();
}

// The k_gemv_ksplit partials for many tokens at once (prefill, state prefill), bit for bit.
// For output (row o, token t) and quarter kq, k_gemv_ksplit lets wave j = 0..15 form
// r_j = MFMA chain over its KPW 32-wide k-blocks (accumulator starting at 0), separately for
// the bf16 hi and lo halves of x (a column of an MFMA result depends only on that column),
// sums r_0 .. r_15 in order, then adds the hi and lo sums. Here one wave walks j = 0..15
// itself with the same operand layout (W rows as A, k slot 8 g + i), so every partial
// coincides. The activations come as bf16 planes from k_split, which rounds as split8_part
// does for finite values. Block: 64 rows x 128 tokens x one k quarter, wave w taking tokens
// 32 w .. 32 w + 31 (two 16-token tiles) for all four row tiles. Used for in = 4096 (KPW 2);
// in = 2048 takes the LDS-tiled k_kva_gemm below.
struct KvaTokArgs {
    float *Y;                  // partial kq at Y + kq * pstride, [S, ldy]
    const uint16_t *XH, *XL;   // [S, in] bf16 hi / lo planes
    const uint16_t *W;         // [out, in]
    size_t pstride;
    int ldy, S, out, in;
};

template <int KPW>
__global__ __launch_bounds__(256) void k_kva_tok(KvaTokArgs a) {
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
    const int kq = blockIdx.y, row0 = blockIdx.x * 64, tok0 = blockIdx.z * 128 + 32 * w;
    const uint16_t *wr[4], *xh[2], *xl[2];
#pragma unroll
    for (int t = 0; t < 4; ++t) wr[t] = a.W + (size_t)min(row0 + 16 * t + n, a.out - 1) * a.in;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const size_t tok = (size_t)min(tok0 + 16 * u + n, a.S - 1);
        xh[u] = a.XH + tok * a.in;
        xl[u] = a.XL + tok * a.in;
    }
    const int kbase = kq * (16 * 32 * KPW) + g * 8;
    v4f sh[4][2], sl[4][2];
    v4i wa[KPW][4], ha[KPW][2], la[KPW][2];
    auto load = [&](int j) {
#pragma unroll
        for (int kb = 0; kb < KPW; ++kb) {
            const int k = kbase + j * (32 * KPW) + 32 * kb;
#pragma unroll
            for (int t = 0; t < 4; ++t) wa[kb][t] = *(const v4i *)(wr[t] + k);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                ha[kb][u] = *(const v4i *)(xh[u] + k);
                la[kb][u] = *(const v4i *)(xl[u] + k);
            }
        }
    };
    load(0);
#pragma unroll 2
    for (int j = 0; j < 16; ++j) {
        v4f rh[4][2], rl[4][2];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                rh[t][u] = v4f{0.f, 0.f, 0.f, 0.f};
                rl[t][u] = v4f{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
        for (int kb = 0; kb < KPW; ++kb)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const v8bf wv = __builtin_bit_cast(v8bf, wa[kb][t]);
                    rh[t][u] = mfma_bf16(wv, __builtin_bit_cast(v8bf, ha[kb][u]), rh[t][u]);
                    rl[t][u] = mfma_bf16(wv, __builtin_bit_cast(v8bf, la[kb][u]), rl[t][u]);
                }
        if (j + 1 < 16) load(j + 1);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                sh[t][u] = j == 0 ? rh[t][u] : sh[t][u] + rh[t][u];
                sl[t][u] = j == 0 ? rl[t][u] : sl[t][u] + rl[t][u];
            }
    }
    float *y = a.Y + (size_t)kq * a.pstride;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int tok = tok0 + 16 * u + n;
        if (tok >= a.S) continue;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const v4f p = sh[t][u] + sl[t][u];
            const int r = row0 + 16 * t + 4 * g;
            float *yp = y + (size_t)tok * a.ldy + r;
            if (r + 3 < a.out && (a.ldy & 3) == 0) {
                *(v4f *)yp = p;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (r + i < a.out) yp[i] = p[i];
            }
        }
    }
}

// The same partials for in = 2048 (one 32-wide k-block per k_gemv_ksplit wave) as a tiled
// GEMM: x hi, x lo and W stream through an LDS ring by DMA (16-byte slot s of a 64-byte
// row r stored at s ^ ((r >> 1) & 3), so the 8 rows of one ds_read_b128 phase hit distinct
// banks). Block: one k quarter of 16 TU WT tokens x 16 TT WR rows, WT x WR waves of TU x TT
// MFMA tiles; per 32-wide k step each tile takes one MFMA from a zero accumulator for the hi
// and one for the lo half, added to the running sums in k order (the sums of k_gemv_ksplit's
// waves 0..15). Tiles are numbered row block fastest, then quarter, then token block, and XCD
// b % 8 takes a contiguous eighth of them, so the row blocks sharing a token block's
// activations run under one L2.
template <int TU_, int TT_, int WT_, int WR_, int NS_>
struct KvgShape {
    static constexpr int TU = TU_, TT = TT_, WT = WT_, WR = WR_, NS = NS_;  // NS: ring stages
    static constexpr int BT = 16 * TU * WT, BR = 16 * TT * WR, NT = 64 * WT * WR;
};

template <class Sh>
__global__ __launch_bounds__(Sh::NT) void k_kva_gemm(KvaTokArgs a) {
    constexpr int TU = Sh::TU, TT = Sh::TT, NS = Sh::NS;
    constexpr int NWV = Sh::WT * Sh::WR, NT = Sh::NT, BT = Sh::BT, BR = Sh::BR;
    constexpr int ROWB = 64, XPL = BT * ROWB, STAGE = 2 * XPL + BR * ROWB;
    constexpr int SLOTS = STAGE / 16, NI = (SLOTS + NT - 1) / NT, NMIN = SLOTS / NT;
    static_assert(SLOTS % 64 == 0 && NS >= 2 && NS <= 16 && NS * STAGE <= 160 * 1024, "the ring is filled by whole waves");
    __shared__ __attribute__((aligned(16))) uint8_t smem[NS * STAGE];
    const uint32_t sbase = lds_addr(smem);
    const int tid = threadIdx.x, l = tid & 63, n = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wt = w % Sh::WT, wr = w / Sh::WT;
    const int nrb = (a.out + BR - 1) / BR, ntb = (a.S + BT - 1) / BT, nt = nrb * kGemvKs * ntb;
    const int xcd = blockIdx.x & 7, rem = nt & 7;
    const int tile = xcd * (nt >> 3) + min(xcd, rem) + (int)(blockIdx.x >> 3);
    const int rb = tile % nrb, kq = (tile / nrb) % kGemvKs, tb = tile / nrb / kGemvKs;
    const int row0 = rb * BR, tok0 = tb * BT;
    auto swz = [](int row) { return (row >> 1) & 3; };
    // DMA: wave w's instruction i fills slots (i * NWV + w) * 64 .. + 63 of a stage: x hi rows,
    // x lo rows, then W rows, 4 slots each. Rows past the end are clamped (never stored).
    const uint8_t *src[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int p = min((i * NWV + w) * 64 + l, SLOTS - 1);
        const int xrow = (p % (BT * 4)) / 4, wrow = (p - 2 * BT * 4) / 4;
        const uint16_t *rp;
        int s;
        if (p < 2 * BT * 4) {
            rp = (p < BT * 4 ? a.XH : a.XL) + (size_t)min(tok0 + xrow, a.S - 1) * a.in;
            s = (p & 3) ^ swz(xrow);
        } else {
            rp = a.W + (size_t)min(row0 + wrow, a.out - 1) * a.in;
            s = (p & 3) ^ swz(wrow);
        }
        src[i] = (const uint8_t *)(rp + kq * 512 + 8 * s);
    }
    auto issue = [&](int j) __attribute__((always_inline)) {
        const uint32_t dst = sbase + (j % NS) * STAGE + (uint32_t)w * 1024;
#pragma unroll
        for (int i = 0; i < NI; ++i)
            if (i < NMIN || (i * NWV + w) * 64 < SLOTS) dma_b128(src[i] + (size_t)j * 64, dst + i * (NWV * 1024));
    };
    int fx[TU], fw[TT];  // fragment offsets: row 16 u + n of the wave's tile, logical slot g
#pragma unroll
    for (int u = 0; u < TU; ++u) {
        const int row = 16 * (TU * wt + u) + n;
        fx[u] = row * ROWB + 16 * (g ^ swz(row));
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int row = 16 * (TT * wr + t) + n;
        fw[t] = 2 * XPL + row * ROWB + 16 * (g ^ swz(row));
    }
    v4f sh[TT][TU], sl[TT][TU];
#pragma unroll
    for (int j = 0; j < NS - 1; ++j) issue(j);
    auto step = [&](int j) __attribute__((always_inline)) {
        // stage j has landed when only the NS - 2 stages after it may still be in flight (a wave
        // issues NMIN or NMIN + 1 copies per stage; waiting for NMIN each is exact or conservative)
        if (j + NS - 1 <= 16) wait_vmcnt<(NS - 2) * NMIN>();
        else wait_vmcnt<0>();
        lds_barrier();  // also: every wave is done with stage j - 1, refilled next
        if (j + NS - 1 < 16) issue(j + NS - 1);
        const uint8_t *st = smem + (j % NS) * STAGE;
        v8bf xh[TU], xl[TU], wv[TT];
#pragma unroll
        for (int u = 0; u < TU; ++u) {
            xh[u] = *(const v8bf *)(st + fx[u]);
            xl[u] = *(const v8bf *)(st + XPL + fx[u]);
        }
#pragma unroll
        for (int t = 0; t < TT; ++t) wv[t] = *(const v8bf *)(st + fw[t]);
        const v4f z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int u = 0; u < TU; ++u) {
                const v4f rh = mfma_bf16(wv[t], xh[u], z);
                const v4f rl = mfma_bf16(wv[t], xl[u], z);
                sh[t][u] = j == 0 ? rh : sh[t][u] + rh;
                sl[t][u] = j == 0 ? rl : sl[t][u] + rl;
            }
    };
    step(0);
#pragma nounroll
    for (int j = 1; j < 16; ++j) step(j);
    float *y = a.Y + (size_t)kq * a.pstride;
    const bool vec = (a.ldy & 3) == 0;
#pragma unroll
    for (int u = 0; u < TU; ++u) {
        const int tok = tok0 + 16 * (TU * wt + u) + n;
        if (tok >= a.S) continue;
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const v4f p = sh[t][u] + sl[t][u];  // lane (g, n): rows 4 g .. 4 g + 3, token n
            const int r = row0 + 16 * (TT * wr + t) + 4 * g;
            float *yp = y + (size_t)tok * a.ldy + r;
            if (vec && r + 3 < a.out) {
                *(v4f *)yp = p;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (r + i < a.out) yp[i] = p[i];
            }
        }
    }
}

template <class Sh>
static hipError_t kva_gemm_launch(hipStream_t st, const KvaTokArgs &a) {
    const size_t tiles = (size_t)((a.out + Sh::BR - 1) / Sh::BR) * kGemvKs * ((a.S + Sh::BT - 1) / Sh::BT);
    if (tiles > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_kva_gemm<Sh>), dim3((unsigned)tiles), dim3(Sh::NT), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_kva_tok(hipStream_t st, float *Y, size_t pstride, int ldy, const uint16_t *XH,
                          const uint16_t *XL, int S, const uint16_t *W, int out, int in) {
    if (!gemv_ksplit_ok(in, in) || S < 1 || out <= 0 || ldy < out || (S + 127) / 128 > 65535 ||
        ((uintptr_t)XH % 16) != 0 || ((uintptr_t)XL % 16) != 0 || ((uintptr_t)W % 16) != 0 ||
        ((uintptr_t)Y % 16) != 0 || pstride % 4 != 0)
        return hipErrorInvalidValue;
    KvaTokArgs a{Y, XH, XL, W, pstride, ldy, S, out, in};
    if (in == 2048) {
        // Small tiles while they do not outnumber the places for them, so that a short prompt spreads
        // over the CUs: first with a ring that holds all 16 k steps (one block per CU; a block then waits
        // for memory about once), then two blocks per CU; large tiles take in fewer bytes per product.
        // us, 32 x 32 and 32 x 64 (16 stages), 32 x 64 (8), 64 x 64, 64 x 96, 128 x 192 (tokens x rows):
        //   37 tokens 5.4 / 6.5 / 6.9 / 9.6 / 11.8 / 17.2   200: 10.3 / 7.2 / 7.4 / 9.9 / - / 19.1
        //   384: 18.5 / 12.5 / 9.2 / 10.3 / - / 19.2        896: 35.7 / 23.9 / 16.5 / 14.3 / - / 20.5
        //   1181: - / - / - / 21.5 / 18.2 / 21.4            16000: - / - / - / - / 171 / 127
        auto tiles = [&](int bt, int br) { return (long)((S + bt - 1) / bt) * kGemvKs * ((out + br - 1) / br); };
        if (tiles(32, 32) <= 256) return kva_gemm_launch<KvgShape<1, 1, 2, 2, 16>>(st, a);
        if (tiles(32, 64) <= 256) return kva_gemm_launch<KvgShape<1, 2, 2, 2, 16>>(st, a);
        if (tiles(32, 64) <= 512) return kva_gemm_launch<KvgShape<1, 2, 2, 2, 8>>(st, a);
        if (tiles(64, 64) <= 512) return kva_gemm_launch<KvgShape<2, 2, 2, 2, 6>>(st, a);
        if (tiles(64, 96) <= 512) return kva_gemm_launch<KvgShape<2, 3, 2, 2, 4>>(st, a);
        return kva_gemm_launch<KvgShape<4, 4, 2, 3, 3>>(st, a);
    } else {
        const dim3 grid((out + 63) / 64, kGemvKs, (S + 127) / 128);
        hipLaunchKernelGGL((k_kva_tok<2>), grid, dim3(256), 0, st, a);
    }
    return hipGetLastError();
}

bool gemv_xs_ok(int in) { return in == 2048 || in == 4096; }

__global__ __launch_bounds__(256) void k_clear_flags(unsigned *zf, int nz) {
    for (int k = threadIdx.x; k < nz; k += 256) *(uint2 *)(zf + (size_t)k * kFqFlagStride) = uint2{0u, 0u};
}
hipError_t launch_clear_flags(hipStream_t st, unsigned *flags, int nlines) {
    hipLaunchKernelGGL(k_clear_flags, dim3(1), dim3(256), 0, st, flags, nlines);
    return hipGetLastError();
}

hipError_t launch_gemv_xs(hipStream_t st, float *Y, int ldy, const uint16_t *XS, int B,
                          const uint16_t *W, int out, int in, bool accumulate, unsigned *zf, int nz) {
    if (!gemv_xs_ok(in) || B < 1 || ((uintptr_t)XS % 16) != 0 || ((uintptr_t)W % 16) != 0 || out <= 0 ||
        (B + 15) / 16 > 65535)
        return hipErrorInvalidValue;
    // 16-token groups of a block: one up to 32 tokens, two in turn beyond (a block's weights serve
    // both). Decodes of 12 layers in turn, kernel trace, two / one group a block (us): 9.7 / 8.0 at 17
    // sequences, 10.1 / 7.7 at 20, 10.8 / 8.0 at 24, 12.2 / 7.7 at 32; at 48, alone, 14.5 / 15.9
    const dim3 grid((out + 15) / 16, 1, B <= 32 ? (B + 15) / 16 : (B + 31) / 32);
    const bool two = B > 8;
    if (in == 2048) {
        // four waves at every batch size: each output is the same sum in the same order whatever
        // the batch (a block decode's members equal lone decodes bit for bit)
        if (two) hipLaunchKernelGGL((k_gemv_xs<2, 16, 16, 4>), grid, dim3(256), 0, st, Y, XS, W, ldy, B, out, in, accumulate ? 1 : 0, zf, nz);
        else hipLaunchKernelGGL((k_gemv_xs<1, 16, 8, 4>), dim3((out + 7) / 8, 1, grid.z), dim3(256), 0, st, Y, XS, W, ldy, B, out, in, accumulate ? 1 : 0, zf, nz);
    } else {
        // eight waves of 16 k-blocks (sixteen waves of 8 spill registers at NG = 2)
        if (two) hipLaunchKernelGGL((k_gemv_xs<2, 16, 16, 8>), grid, dim3(512), 0, st, Y, XS, W, ldy, B, out, in, accumulate ? 1 : 0, zf, nz);
        else hipLaunchKernelGGL((k_gemv_xs<1, 16, 16, 8>), grid, dim3(512), 0, st, Y, XS, W, ldy, B, out, in, accumulate ? 1 : 0, zf, nz);
    }
    return hipGetLastError();
}

hipError_t launch_gemv(hipStream_t st, float *Y, int ldy, const float *X, int ldx, int B,
                       const uint16_t *W0, int out0, const uint16_t *W1, int out1, int in,
                       bool accumulate) {
    GemvArgs a{Y, X, W0, W1, ldy, ldx, B, out0, out1, in, accumulate ? 1 : 0};
    const int out = out0 + out1;
    if (out <= 0 || B <= 0) return hipSuccess;
    const bool aligned = (in % 256) == 0 && (ldx % 4) == 0 && ((uintptr_t)X % 16) == 0 &&
                         ((uintptr_t)W0 % 16) == 0 && (!W1 || ((uintptr_t)W1 % 16) == 0);
    if (aligned) {
        dim3 grid((out + 15) / 16, (B + 15) / 16);
        if (in % 512 == 0) hipLaunchKernelGGL(k_gemv_mfma<16>, grid, dim3(1024), 0, st, a);
        else hipLaunchKernelGGL(k_gemv_mfma<8>, grid, dim3(512), 0, st, a);
    } else {
        hipLaunchKernelGGL(k_gemv_generic, dim3((out + 3) / 4), dim3(256), 0, st, a);
    }
    return hipGetLastError();
}

// ================================================================ append ===============

constexpr int kMaxR = 1024;   // kv_lora_rank bound of the device kernels
constexpr int kMaxDR = 256;   // qk_rope_dim bound
constexpr int kMaxDN = 512;   // qk_nope_dim bound

// The sequence table and dims are separate kernel arguments (one copy serves the fused
// append + qprep launch).
struct AppendArgs {
    const float *y;  // projection rows: np partials pstride apart, summed in order
    const uint16_t *norm;
    const float2 *cs;
    uint8_t *rows;
    float *latent;
    size_t pstride;
    int ldy, koff, np, fmt, normed, row_bytes, rows_mode;
    float eps;
};

// Sequence descriptors without a read that waits on the sequence index: lane i of a fully
// active wave reads descriptor i of the table (kernel arguments, kMaxBatch = 64 = one entry per
// lane) in the first round trip beside the other arguments, and the wave then takes the entry
// of a wave-uniform index from that lane. Indexing the table once the index is known costs one
// more memory round trip.
static_assert(kMaxBatch == 64, "one descriptor per lane");
__device__ __forceinline__ int lane_pick(int v, int b) { return __builtin_amdgcn_readlane(v, b); }
__device__ __forceinline__ void *lane_pick(void *p, int b) {
    const uint64_t u = (uint64_t)p;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, b);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), b);
    return (void *)(((uint64_t)hi << 32) | lo);
}
struct DescLane {  // this lane's entry of the table
    void *a, *b, *c;
    int len, pos, split0, nsplit, rps;
};
__device__ __forceinline__ DescLane desc_lane(const SeqTable &t) {
    const SeqDesc &m = t.s[threadIdx.x & 63];
    return DescLane{m.a, m.b, m.c, m.len, m.pos, m.split0, m.nsplit, m.rps};
}
__device__ __forceinline__ SeqDesc desc_pick(const DescLane &m, int i) {
    SeqDesc s;
    s.a = lane_pick(m.a, i);
    s.b = lane_pick(m.b, i);
    s.c = lane_pick(m.c, i);
    s.len = lane_pick(m.len, i);
    s.pos = lane_pick(m.pos, i);
    s.split0 = lane_pick(m.split0, i);
    s.nsplit = lane_pick(m.nsplit, i);
    s.rps = lane_pick(m.rps, i);
    s.pad1 = 0;
    return s;
}

// Value of a projection output stored as np partials (np = 1 or kGemvKs) pstride floats
// apart, added in partial order. The kGemvKs loads are issued together.
__device__ __forceinline__ float sum_parts(const float *p, int np, size_t pstride) {
    if (np == kGemvKs) {
        float v[kGemvKs];
#pragma unroll
        for (int q = 0; q < kGemvKs; ++q) v[q] = p[(size_t)q * pstride];
        float s = v[0];
#pragma unroll
        for (int q = 1; q < kGemvKs; ++q) s += v[q];
        return s;
    }
    return p[0];
}

// One block per sequence (rows_mode = 0) or, with rows_mode = 1, one block per row of the
// single sequence t.s[0]: block i appends row t.s[0].pos + i from input row i. Reproduces src/ops.c:76-83 (RMSNorm: double sum of squares,
// inv = 1/sqrtf(float(ss/n) + eps), (x*inv)*w), src/mla_compressed_q8_state.c:34-55
// (absmax/127, inv = 1/scale, roundf, clamp) and the RoPE rotation of
// src/mla_compressed_q8_state.c:18-32 with host-computed (cos, sin) pairs. The library is
// compiled with -ffp-contract=off, so each product and sum rounds separately as there.
__device__ __forceinline__ void append_body(const SeqTable &t, const Dims &d, const AppendArgs &a, int b) {
    __shared__ float lat[kMaxR];
    __shared__ float kat[kMaxR + kMaxDR];  // projection row: RMSNorm input | RoPE input
    __shared__ double redd[4];
    __shared__ float redf[4];
    const int tid = threadIdx.x;
    const SeqDesc s = desc_pick(desc_lane(t), a.rows_mode ? 0 : b);
    const int R = d.R, DR = d.DR, half = DR / 2, pos = s.pos + (a.rows_mode ? b : 0);
    const int nk = R + DR;
    const float *ky = a.y + (size_t)b * a.ldy + a.koff;
    // All global reads first, so that one memory round trip covers them: the projection row
    // (partials summed), the norm weights of this thread's first two columns, its RoPE pair.
    float kv[3], nw[2];
#pragma unroll
    for (int j = 0; j < 3; ++j) kv[j] = sum_parts(ky + min(tid + 256 * j, nk - 1), a.np, a.pstride);
#pragma unroll
    for (int j = 0; j < 2; ++j) nw[j] = a.normed ? 0.f : bf16_to_f32(a.norm[min(tid + 256 * j, R - 1)]);
    const float2 csv = half > 0 ? a.cs[(size_t)pos * half + min(tid, half - 1)] : float2{0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 3; ++j)
        if (tid + 256 * j < nk) kat[tid + 256 * j] = kv[j];
    for (int r = tid + 768; r < nk; r += 256) kat[r] = sum_parts(ky + r, a.np, a.pstride);  // R + DR > 768
    __syncthreads();

    if (!a.normed) {
        double ss = 0.0;
        for (int r = tid; r < R; r += 256) {
            const double v = (double)kat[r];
            ss += v * v;
        }
        const float mean_sq = (float)(block256_sum_f64(ss, redd) / (double)R);
        const float inv = 1.0f / sqrtf(mean_sq + a.eps);
        for (int r = tid, j = 0; r < R; r += 256, ++j) {
            const float t = kat[r] * inv;
            lat[r] = t * (j < 2 ? nw[j] : bf16_to_f32(a.norm[r]));
        }
    } else {
        for (int r = tid; r < R; r += 256) lat[r] = kat[r];
    }
    __syncthreads();

    uint8_t *row_out = a.rows + (size_t)b * a.row_bytes;
    if (a.fmt == kFmtQ8) {
        float m = 0.f;
        for (int r = tid; r < R; r += 256) m = fmaxf(m, fabsf(lat[r]));
        // fmaxf drops NaN operands: a NaN latent must still select the zero row, as the
        // reference's sequential `a > amax` scan followed by isfinite() does for Inf; NaN
        // never compares greater there, so it is simply skipped -- identical to fmaxf.
        const float amax = block256_max(m, redf);
        int8_t *codes = (int8_t *)s.a + (size_t)pos * R;
        const bool zero = !(amax > 0.0f) || !isfinite(amax);
        const float scale = zero ? 1.0f : amax / 127.0f;
        const float inv = zero ? 0.0f : 1.0f / scale;
        for (int r = tid; r < R; r += 256) {
            int8_t q = 0;
            if (!zero) {
                float v = roundf(lat[r] * inv);
                v = v > 127.0f ? 127.0f : v;
                v = v < -127.0f ? -127.0f : v;
                q = (int8_t)v;
            }
            codes[r] = q;
            row_out[r] = (uint8_t)q;
        }
        if (tid == 0) {
            ((float *)s.b)[pos] = scale;
            *(float *)(row_out + R) = scale;
        }
    } else if (a.fmt == kFmtF32) {
        float *dst = (float *)s.a + (size_t)pos * R;
        for (int r = tid; r < R; r += 256) {
            dst[r] = lat[r];
            ((float *)row_out)[r] = lat[r];
        }
    } else if (a.fmt == kFmtBF16) {
        uint16_t *dst = (uint16_t *)s.a + (size_t)pos * R;
        for (int r = tid; r < R; r += 256) {
            const uint16_t h = f32_to_bf16_rne(lat[r]);
            dst[r] = h;
            ((uint16_t *)row_out)[r] = h;
        }
    } else {
        for (int r = tid; r < R; r += 256) a.latent[(size_t)b * R + r] = lat[r];
    }

    if (tid < half) {  // half <= kMaxDR / 2 < 256
        const int i = tid;
        const float2 cs = csv;
        const float ev = kat[R + 2 * i], od = kat[R + 2 * i + 1];
        const float ec = ev * cs.x, os = od * cs.y, oc = od * cs.x, es = ev * cs.y;
        const float d0 = ec - os, d1 = oc + es;
        if (a.fmt == kFmtQ8) {
            uint16_t *rp = (uint16_t *)s.c + (size_t)pos * DR;
            const uint16_t h0 = f32_to_bf16_rne(d0), h1 = f32_to_bf16_rne(d1);
            rp[i] = h0;
            rp[half + i] = h1;
            uint16_t *ro = (uint16_t *)(row_out + R + 4);
            ro[i] = h0;
            ro[half + i] = h1;
        } else if (a.fmt == kFmtF32) {
            float *rp = (float *)s.b + (size_t)pos * DR;
            rp[i] = d0;
            rp[half + i] = d1;
            float *ro = (float *)row_out + R;
            ro[i] = d0;
            ro[half + i] = d1;
        } else if (a.fmt == kFmtBF16) {
            uint16_t *rp = (uint16_t *)s.b + (size_t)pos * DR;
            const uint16_t h0 = f32_to_bf16_rne(d0), h1 = f32_to_bf16_rne(d1);
            rp[i] = h0;
            rp[half + i] = h1;
            uint16_t *ro = (uint16_t *)row_out + R;
            ro[i] = h0;
            ro[half + i] = h1;
        } else {
            float *ro = (float *)row_out;  // expanded: rotated key staged for store_expanded
            ro[i] = d0;
            ro[half + i] = d1;
        }
    }
}

__global__ __launch_bounds__(256) void k_append(SeqTable t, Dims d, AppendArgs a) {
    append_body(t, d, a, blockIdx.x);
}

// Rows mode of k_append for R = 512, DR = 64 (Q8, FP32, BF16 rows), one wave per row: lane l holds
// columns l + 64 q and does the arithmetic of k_append's threads l + 64 w (their sums of squares per
// former wave, then the four sums in its order), so the rows are k_append's bit for bit, without its
// barriers and with every load of a row requested at once. stage: also write the copy at a.rows.
// k_append waited through four dependent phases per row. Fills of a state on the device, where nobody
// reads the copy: 16000 BF16 rows 57 -> 41 us (165 MB, most of it the four partials), 1181 Q8 rows
// 7.2 -> 5.2.
template <int FMT>
__global__ __launch_bounds__(256) void k_append_rows(SeqDesc s, AppendArgs a, int nrows, int stage) {
    constexpr int R = 512, DR = 64;
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    float nw[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) nw[q] = bf16_to_f32(a.norm[l + 64 * q]);
    for (int b = blockIdx.x * 4 + w; b < nrows; b += gridDim.x * 4) {
        const int pos = s.pos + b;
        const float *ky = a.y + (size_t)b * a.ldy + a.koff + l;
        float kv[9];
#pragma unroll
        for (int q = 0; q < 9; ++q) kv[q] = sum_parts(ky + 64 * q, kGemvKs, a.pstride);
        const float2 cs = a.cs[(size_t)pos * 32 + (l & 31)];
        double sw[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const double v0 = (double)kv[i], v1 = (double)kv[i + 4];
            double ss = v0 * v0;
            ss += v1 * v1;
            sw[i] = wave_sum_f64(ss);
        }
        const float mean_sq = (float)(((sw[0] + sw[1]) + (sw[2] + sw[3])) / (double)R);
        const float inv = 1.0f / sqrtf(mean_sq + a.eps);
        float lat[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const float t = kv[q] * inv;
            lat[q] = t * nw[q];
        }
        // rotated key: lane i < 32 takes pair i
        const float ev = __shfl(kv[8], 2 * (l & 31)), od = __shfl(kv[8], 2 * (l & 31) + 1);
        const float ec = ev * cs.x, os = od * cs.y, oc = od * cs.x, es = ev * cs.y;
        const float key = l < 32 ? ec - os : oc + es;  // element l
        uint8_t *row_out = a.rows + (size_t)b * a.row_bytes;
        if constexpr (FMT == kFmtQ8) {
            float m = 0.f;
#pragma unroll
            for (int q = 0; q < 8; ++q) m = fmaxf(m, fabsf(lat[q]));  // drops NaN, as k_append's
            const float amax = wave_max(m);
            int8_t *codes = (int8_t *)s.a + (size_t)pos * R;
            const bool zero = !(amax > 0.0f) || !isfinite(amax);
            const float scale = zero ? 1.0f : amax / 127.0f;
            const float qi = zero ? 0.0f : 1.0f / scale;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                int8_t c = 0;
                if (!zero) {
                    float v = roundf(lat[q] * qi);
                    v = v > 127.0f ? 127.0f : v;
                    v = v < -127.0f ? -127.0f : v;
                    c = (int8_t)v;
                }
                codes[l + 64 * q] = c;
                if (stage) row_out[l + 64 * q] = (uint8_t)c;
            }
            const uint16_t h = f32_to_bf16_rne(key);
            ((uint16_t *)s.c)[(size_t)pos * DR + l] = h;
            if (stage) ((uint16_t *)(row_out + R + 4))[l] = h;
            if (l == 0) {
                ((float *)s.b)[pos] = scale;
                if (stage) *(float *)(row_out + R) = scale;
            }
        } else if constexpr (FMT == kFmtF32) {
            float *dst = (float *)s.a + (size_t)pos * R;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                dst[l + 64 * q] = lat[q];
                if (stage) ((float *)row_out)[l + 64 * q] = lat[q];
            }
            ((float *)s.b)[(size_t)pos * DR + l] = key;
            if (stage) ((float *)row_out)[R + l] = key;
        } else {
            uint16_t *dst = (uint16_t *)s.a + (size_t)pos * R;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const uint16_t h = f32_to_bf16_rne(lat[q]);
                dst[l + 64 * q] = h;
                if (stage) ((uint16_t *)row_out)[l + 64 * q] = h;
            }
            const uint16_t h = f32_to_bf16_rne(key);
            ((uint16_t *)s.b)[(size_t)pos * DR + l] = h;
            if (stage) ((uint16_t *)row_out)[R + l] = h;
        }
    }
}

static AppendArgs append_args(int fmt, const Dims &d, const float *y, int ldy, int koff,
                              int ynp, size_t ypstride, const uint16_t *kv_a_norm, float eps,
                              const float2 *rope_cs, const DecodeWork &w, bool normed, int nrows) {
    AppendArgs a;
    a.y = y;
    a.np = ynp > 1 ? ynp : 1;
    a.pstride = ypstride;
    a.norm = kv_a_norm;
    a.cs = rope_cs;
    a.rows = w.rows;
    a.latent = w.latent;
    a.ldy = ldy;
    a.koff = koff;
    a.fmt = fmt;
    a.normed = normed ? 1 : 0;
    a.row_bytes = fmt == kFmtQ8    ? d.R + 4 + 2 * d.DR
                  : fmt == kFmtF32 ? 4 * (d.R + d.DR)
                  : fmt == kFmtBF16 ? 2 * (d.R + d.DR)
                                    : 4 * d.NH * (d.QD + d.DV);
    a.eps = eps;
    a.rows_mode = nrows > 0 ? 1 : 0;
    return a;
}

hipError_t launch_append(hipStream_t st, int fmt, const SeqTable &t, const Dims &d,
                         const float *y, int ldy, int koff, int ynp, size_t ypstride,
                         const uint16_t *kv_a_norm, float eps, const float2 *rope_cs,
                         const DecodeWork &w, bool normed, int nrows, bool stage) {
    if (d.R > kMaxR || d.DR > kMaxDR || (ynp != 1 && ynp != kGemvKs)) return hipErrorInvalidValue;
    const AppendArgs a = append_args(fmt, d, y, ldy, koff, ynp, ypstride, kv_a_norm, eps, rope_cs, w,
                                     normed, nrows);
    if (nrows > 0 && d.R == 512 && d.DR == 64 && ynp == kGemvKs && !normed && fmt != kFmtExp) {
        const dim3 grid(std::min((nrows + 3) / 4, 2048));  // eight blocks a CU, rows in turn beyond
        if (fmt == kFmtQ8) hipLaunchKernelGGL(k_append_rows<kFmtQ8>, grid, dim3(256), 0, st, t.s[0], a, nrows, stage ? 1 : 0);
        else if (fmt == kFmtF32) hipLaunchKernelGGL(k_append_rows<kFmtF32>, grid, dim3(256), 0, st, t.s[0], a, nrows, stage ? 1 : 0);
        else hipLaunchKernelGGL(k_append_rows<kFmtBF16>, grid, dim3(256), 0, st, t.s[0], a, nrows, stage ? 1 : 0);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_append, dim3(nrows > 0 ? nrows : t.n), dim3(256), 0, st, t, d, a);
    return hipGetLastError();
}

// y = x * (1/sqrtf(float(sum x^2 / n) + eps)) * w for `rows` rows of length n
// (src/ops.c:76-83). Double sum of squares in a fixed per-thread-then-tree order.
__global__ __launch_bounds__(256) void k_rmsnorm(float *y, const float *x, const uint16_t *wt,
                                                 int n, float eps) {
    __shared__ double redd[256];
    const int tid = threadIdx.x;
    const float *xr = x + (size_t)blockIdx.x * n;
    float *yr = y + (size_t)blockIdx.x * n;
    double ss = 0.0;
    for (int i = tid; i < n; i += 256) {
        const double v = (double)xr[i];
        ss += v * v;
    }
    redd[tid] = ss;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) redd[tid] += redd[tid + o];
        __syncthreads();
    }
    const float mean_sq = (float)(redd[0] / (double)n);
    const float inv = 1.0f / sqrtf(mean_sq + eps);
    for (int i = tid; i < n; i += 256) {
        const float t = xr[i] * inv;
        yr[i] = t * bf16_to_f32(wt[i]);
    }
}

// The same for n <= 256 NV with every load requested up front (x and weights in registers): the loop
// of k_rmsnorm waits for each of its loads in turn, and its tree for eight barriers. The same values
// are added in the same order (thread sums, halves of 128 and 64, then the lanes of a wave), so the
// results are those of k_rmsnorm bit for bit. 8 rows of 2048, two launches per layer of the decode
// stack: 6.3 -> 4.7 us per launch (kernel trace), 27 layers 1.73 -> 1.52 ms; bound by two memory
// round trips and the launch itself.
template <int NV>
__global__ __launch_bounds__(256) void k_rmsnorm_reg(float *y, const float *x, const uint16_t *wt, int n, float eps) {
    __shared__ double redd[256];
    const int tid = threadIdx.x, l = tid & 63;
    const float *xr = x + (size_t)blockIdx.x * n;
    float *yr = y + (size_t)blockIdx.x * n;
    float v[NV];
    uint16_t w[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int k = min(tid + 256 * i, n - 1);
        v[i] = xr[k];
        w[i] = wt[k];
    }
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const double d = tid + 256 * i < n ? (double)v[i] : 0.0;
        ss += d * d;
    }
    redd[tid] = ss;
    __syncthreads();
    double t = (redd[l] + redd[l + 128]) + (redd[l + 64] + redd[l + 192]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o);
    const float mean_sq = (float)(lane_f64(t, 0) / (double)n);
    const float inv = 1.0f / sqrtf(mean_sq + eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const float u = v[i] * inv;
        if (tid + 256 * i < n) yr[tid + 256 * i] = u * bf16_to_f32(w[i]);
    }
}

hipError_t launch_rmsnorm(hipStream_t st, float *y, const float *x, const uint16_t *w, int n,
                          int rows, float eps) {
    if (rows <= 0 || n <= 0) return hipSuccess;
    if (n <= 256 * 8) hipLaunchKernelGGL((k_rmsnorm_reg<8>), dim3(rows), dim3(256), 0, st, y, x, w, n, eps);
    else if (n <= 256 * 16) hipLaunchKernelGGL((k_rmsnorm_reg<16>), dim3(rows), dim3(256), 0, st, y, x, w, n, eps);
    else hipLaunchKernelGGL(k_rmsnorm, dim3(rows), dim3(256), 0, st, y, x, w, n, eps);
    return hipGetLastError();
}

// Expanded state: K = [kv_b(latent)[h, :DN] | rotated key], V = kv_b(latent)[h, DN:]
// (src/mla_state.c:95-115). One block per sequence; rows staged for host write-back.
struct StoreExpArgs {
    SeqTable t;
    Dims d;
    const float *kv;
    uint8_t *rows;
};

__global__ __launch_bounds__(256) void k_store_expanded(StoreExpArgs a) {
    const int b = blockIdx.x, tid = threadIdx.x;
    const SeqDesc &s = a.t.s[b];
    const Dims &d = a.d;
    const size_t row_bytes = (size_t)4 * d.NH * (d.QD + d.DV);
    float *stage = (float *)(a.rows + (size_t)b * row_bytes);
    // the rotated key was staged by k_append at the front of this sequence's row slot
    __shared__ float rope[kMaxDR];
    for (int i = tid; i < d.DR; i += 256) rope[i] = stage[i];
    __syncthreads();
    float *keys = (float *)s.a + (size_t)s.pos * d.NH * d.QD;
    float *vals = (float *)s.b + (size_t)s.pos * d.NH * d.DV;
    const float *kv = a.kv + (size_t)b * d.KVB;
    const int nk = d.NH * d.QD, nv = d.NH * d.DV;
    for (int i = tid; i < nk; i += 256) {
        const int h = i / d.QD, k = i % d.QD;
        keys[i] = k < d.DN ? kv[h * (d.DN + d.DV) + k] : rope[k - d.DN];
    }
    for (int i = tid; i < nv; i += 256) {
        const int h = i / d.DV, k = i % d.DV;
        vals[i] = kv[h * (d.DN + d.DV) + d.DN + k];
    }
    __syncthreads();
    for (int i = tid; i < nk; i += 256) stage[i] = keys[i];
    for (int i = tid; i < nv; i += 256) stage[nk + i] = vals[i];
}

hipError_t launch_store_expanded(hipStream_t st, const SeqTable &t, const Dims &d,
                                 const DecodeWork &w) {
    if (d.DR > kMaxDR) return hipErrorInvalidValue;
    StoreExpArgs a{t, d, w.kv, w.rows};
    hipLaunchKernelGGL(k_store_expanded, dim3(t.n), dim3(256), 0, st, a);
    return hipGetLastError();
}

// ================================================================ query prep ===========

// W_UK^T in the order the query preparation's MFMA A operands are loaded (R = 512, DN = 128):
// fragment (head h, wave w, tile t, k-step ks) is 64 lanes x 16 bytes, contiguous, lane l holding
// W_UK[d = 32 ks + 8 (l >> 4) + e, latent column j = 128 w + 16 t + (l & 15)], e = 0..7, where
// W_UK[d, j] = kv_b[h * (DN + DV) + d, j]. One load instruction then reads 1 KB in one run. One
// thread per output element.
__global__ __launch_bounds__(256) void k_wuk_t(uint16_t *dst, const uint16_t *kv_b, int NH, int DN, int DV, int R) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, n = (size_t)NH * R * DN;
    if (i >= n) return;
    const int e = (int)(i & 7), l = (int)((i >> 3) & 63), ks = (int)((i >> 9) & 3), t = (int)((i >> 11) & 7),
              w = (int)((i >> 14) & 3), h = (int)(i >> 16);
    const int dd = 32 * ks + 8 * (l >> 4) + e, j = 128 * w + 16 * t + (l & 15);
    dst[i] = kv_b[((size_t)h * (DN + DV) + dd) * R + j];
}

hipError_t launch_wuk_transpose(hipStream_t st, uint16_t *dst, const uint16_t *kv_b, const Dims &d) {
    if (d.R != 512 || d.DN != 128) return hipErrorInvalidValue;
    const size_t n = (size_t)d.NH * d.R * d.DN;
    hipLaunchKernelGGL(k_wuk_t, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dst, kv_b, d.NH, d.DN, d.DV, d.R);
    return hipGetLastError();
}

struct QprepArgs {
    const float *y;  // projection rows: np partials pstride apart, summed in order
    const uint16_t *kv_b;
    const uint16_t *ukt;  // W_UK^T [NH, R, DN] bf16 (the MFMA operand of the Kimi-shape path) or null
    const float2 *cs;
    float *qf;
    int8_t *qhi, *qlo;
    float *qs;
    uint16_t *qrhi, *qrlo;
    size_t pstride;
    int ldy, np, fmt, quantize;
    int quarter;  // fp32 query rows by qprep_quarter (compressed formats, R = 512, DN = 128, DR = 64)
};

// One block per (sequence, head). Compressed formats: q_lat[r] = sum_d
// kv_b[h*(DN+DV)+d, r] * q_nope[d] (src/mla_compressed_q8_state.c:206-214), q_rope rotated
// at the decode position; qf row = [q_lat | q_rope]. Expanded: qf row = [q_nope | q_rope].
// With `quantize`, q_lat ~= qs * (hi + lo/254) (int8 hi, lo) and q_rope / sqrt(QD) = hi + lo
// (bf16).
__device__ __forceinline__ void qprep_body(const SeqTable &t, const Dims &d, const QprepArgs &a, int blk) {
    __shared__ __attribute__((aligned(16))) float qn[kMaxDN];
    __shared__ float qr[kMaxDR];  // RoPE input of the head
    __shared__ float ql[kMaxR];
    __shared__ float redf[4];
    const DescLane dl = desc_lane(t);
    const int b = blk / d.NH, h = blk % d.NH, tid = threadIdx.x;
    const SeqDesc s = desc_pick(dl, b);
    const float *qh = a.y + (size_t)b * a.ldy + (size_t)h * d.QD;
    const int half = d.DR / 2, nq = d.DN + d.DR;
    // Kimi shapes: q_lat = W_UK^T q_nope on MFMA. Wave w owns latent columns 128 w .. +127 as
    // eight 16-column tiles; the A operands come from the copy of W_UK^T made with the weights,
    // stored in fragment order (k_wuk_t): lane (g, n) of fragment (t, ks) holds latent column
    // 128 w + 16 t + n, d = 32 ks + 8 g .. +7. Requested before q since they do not depend on it.
    const bool fast = a.fmt != kFmtExp && d.R == 512 && d.DN == 128 && a.ukt != nullptr;
    v8bf wa[8][4];
    if (fast) {
        const uint16_t *ut = a.ukt + ((size_t)(h * 4 + (tid >> 6)) * 32 * 64 + (tid & 63)) * 8;
#pragma unroll
        for (int t = 0; t < 8; ++t)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) wa[t][ks] = *(const v8bf *)(ut + (size_t)(t * 4 + ks) * 64 * 8);
    }
    // the query head (partials summed) and this thread's RoPE pair, in one round trip
    {
        const float v = sum_parts(qh + min(tid, nq - 1), a.np, a.pstride);
        if (tid < d.DN) qn[tid] = v;
        else if (tid < nq) qr[tid - d.DN] = v;
        for (int i = tid + 256; i < nq; i += 256) {  // DN + DR > 256
            const float u = sum_parts(qh + i, a.np, a.pstride);
            if (i < d.DN) qn[i] = u;
            else qr[i - d.DN] = u;
        }
    }
    const float2 csv = half > 0 ? a.cs[(size_t)s.pos * half + min(tid, half - 1)] : float2{0.f, 0.f};
    __syncthreads();
    const bool exp = a.fmt == kFmtExp;
    const int qstride = exp ? d.QD : d.R + d.DR;
    const int roff = exp ? d.DN : d.R;
    float *qrow = a.qf + ((size_t)b * d.NH + h) * qstride;
    if (exp) {
        for (int i = tid; i < d.DN; i += 256) qrow[i] = qn[i];
    } else {
        const uint16_t *wuk = a.kv_b + (size_t)h * (d.DN + d.DV) * d.R;
        if (fast) {
            // B operand: column 0 = bf16 hi of q_nope, column 1 = its lo part (hi + lo keeps ~16
            // bits; the products are exact in the fp32 accumulator), columns 2-15 zero. D row
            // 4 g + i of tile t is latent column 128 w + 16 t + 4 g + i; columns 0 and 1 (lanes
            // n = 0, 1) are added by one DPP swap.
            const int w = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
            // every lane splits its 8 values (no divergence), lanes n = 0 / 1 keep hi / lo
            const int m0 = n == 0 ? -1 : 0, m1 = n == 1 ? -1 : 0;
            v8bf qb[4];
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const v4f x0 = *(const v4f *)(qn + 32 * ks + 8 * g), x1 = *(const v4f *)(qn + 32 * ks + 8 * g + 4);
                v8bf hi, lo;
                split8_cvt(x0, x1, hi, lo);
                const v4i hv = __builtin_bit_cast(v4i, hi), lv = __builtin_bit_cast(v4i, lo);
                qb[ks] = __builtin_bit_cast(v8bf, (hv & m0) | (lv & m1));
            }
            v4f acc[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) acc[t] = mfma_bf16(wa[t][ks], qb[ks], acc[t]);
            }
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                v4f v;
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = acc[t][i] + dpp_f32<0xB1>(acc[t][i]);  // quad_perm [1,0,3,2]
                if (n == 0) {
                    const int r = 128 * w + 16 * t + 4 * g;
#pragma unroll
                    for (int i = 0; i < 4; ++i) ql[r + i] = v[i];
                    *(v4f *)(qrow + r) = v;
                }
            }
        } else if ((d.R & 1) == 0) {
            // two adjacent latent columns per thread (one 4-byte load per k), 4 k in flight
            for (int r = 2 * tid; r < d.R; r += 512) {
                float a0 = 0.f, a1 = 0.f, b0 = 0.f, b1 = 0.f;
                int k = 0;
                for (; k + 2 <= d.DN; k += 2) {
                    const uint32_t u0 = *(const uint32_t *)(wuk + (size_t)k * d.R + r);
                    const uint32_t u1 = *(const uint32_t *)(wuk + (size_t)(k + 1) * d.R + r);
                    a0 = fmaf(__uint_as_float(u0 << 16), qn[k], a0);
                    a1 = fmaf(__uint_as_float(u0 & 0xffff0000u), qn[k], a1);
                    b0 = fmaf(__uint_as_float(u1 << 16), qn[k + 1], b0);
                    b1 = fmaf(__uint_as_float(u1 & 0xffff0000u), qn[k + 1], b1);
                }
                for (; k < d.DN; ++k) {
                    const uint32_t u0 = *(const uint32_t *)(wuk + (size_t)k * d.R + r);
                    a0 = fmaf(__uint_as_float(u0 << 16), qn[k], a0);
                    a1 = fmaf(__uint_as_float(u0 & 0xffff0000u), qn[k], a1);
                }
                ql[r] = a0 + b0;
                ql[r + 1] = a1 + b1;
                qrow[r] = a0 + b0;
                qrow[r + 1] = a1 + b1;
            }
        } else {
            for (int r = tid; r < d.R; r += 256) {
                float acc = 0.f;
                for (int k = 0; k < d.DN; ++k) acc = fmaf(bf16_to_f32(wuk[(size_t)k * d.R + r]), qn[k], acc);
                ql[r] = acc;
                qrow[r] = acc;
            }
        }
    }
    if (tid < half) {  // half <= kMaxDR / 2 < 256
        const int i = tid;
        const float2 cs = csv;
        const float ev = qr[2 * i], od = qr[2 * i + 1];
        const float ec = ev * cs.x, os = od * cs.y, oc = od * cs.x, es = ev * cs.y;
        const float r0 = ec - os, r1 = oc + es;
        qrow[roff + i] = r0;
        qrow[roff + half + i] = r1;
        if (a.quantize) {
            // the bf16 hi/lo operands of the Q8 attention carry the softmax scale 1/sqrt(QD)
            uint16_t hi, lo;
            const size_t o = ((size_t)b * d.NH + h) * d.DR;
            const float qsc = 1.0f / sqrtf((float)d.QD);
            split_bf16(r0 * qsc, hi, lo);
            a.qrhi[o + i] = hi;
            a.qrlo[o + i] = lo;
            split_bf16(r1 * qsc, hi, lo);
            a.qrhi[o + half + i] = hi;
            a.qrlo[o + half + i] = lo;
        }
    }
    if (!a.quantize || exp) return;
    __syncthreads();
    float m = 0.f;
    for (int r = tid; r < d.R; r += 256) m = fmaxf(m, fabsf(ql[r]));
    const float amax = block256_max(m, redf);
    const bool ok = amax > 0.f && isfinite(amax);
    const float inv = ok ? 127.0f / amax : 0.f;
    const size_t o = ((size_t)b * d.NH + h) * d.R;
    for (int r = tid; r < d.R; r += 256) {
        const float v = ql[r] * inv;
        float hi = rintf(v);
        hi = fminf(fmaxf(hi, -127.f), 127.f);
        float lo = rintf((v - hi) * 254.0f);  // |v - hi| <= 1/2: lo spans the int8 range
        lo = fminf(fmaxf(lo, -127.f), 127.f);
        a.qhi[o + r] = (int8_t)hi;
        a.qlo[o + r] = (int8_t)lo;
    }
    if (tid == 0) a.qs[(size_t)b * d.NH + h] = ok ? amax / 127.0f : 0.f;
}

// The fp32 query rows (the operands of the BF16 and FP32 attention and of the generic path)
// for R = 512, DN = 128, DR = 64, a quarter of the latent columns per block: block (g8, h, qq)
// prepares head h of the (up to) 8 sequences 8 g8 .. 8 g8 + 7 for latent columns 128 qq .. +127,
// taking in a quarter of W_UK^T (32 KB) instead of all of it (qprep_body: one block per
// sequence and head). q_lat = W_UK^T q_nope on MFMA with the 16 B-operand columns holding the
// bf16 hi (0-7) and lo (8-15) parts of the 8 sequences' q_nope: every output element is the
// same product chain as in qprep_body (hi column + lo column, k-steps in order), so the rows
// are bit-identical to it. Wave w owns latent columns 128 qq + 32 w .. + 31 (W_UK^T fragments
// (h, qq, 2w + t, ks)). The quarter-0 blocks also rotate q_rope (one pair per thread).
__device__ __forceinline__ void qprep_quarter(const SeqTable &t, const QprepArgs &a, int blk, int NH) {
    __shared__ __attribute__((aligned(16))) float qn8[8][132];  // q_nope of the 8 sequences
    const DescLane dl = desc_lane(t);
    const int g8 = blk / (NH * 4), h = (blk / 4) % NH, qq = blk & 3;
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
    const int nseq = min(8, t.n - 8 * g8);
    v8bf wa[2][4];
    {
        const uint16_t *ut = a.ukt + ((size_t)((h * 4 + qq) * 8 + 2 * w) * 4 * 64 + l) * 8;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) wa[tt][ks] = *(const v8bf *)(ut + (size_t)(tt * 4 + ks) * 64 * 8);
    }
    // q_nope of sequence js = tid / 32, dims 4 (tid % 32) .. + 3: the partials added in order
    const int js = tid >> 5, b = 8 * g8 + min(js, nseq - 1);
    const float *qh = a.y + (size_t)b * a.ldy + (size_t)h * 192;
    {
        const float *p = qh + 4 * (tid & 31);
        v4f v = *(const v4f *)p;
        if (a.np == kGemvKs) {
            v4f u[kGemvKs - 1];
#pragma unroll
            for (int q = 1; q < kGemvKs; ++q) u[q - 1] = *(const v4f *)(p + (size_t)q * a.pstride);
#pragma unroll
            for (int q = 1; q < kGemvKs; ++q) v += u[q - 1];
        }
        *(v4f *)&qn8[js][4 * (tid & 31)] = v;
    }
    // q_rope pair i = tid % 32 of sequence js (quarter-0 blocks)
    float ev = 0.f, od = 0.f;
    float2 cs = {0.f, 0.f};
    if (qq == 0) {
        const int i = tid & 31;
        ev = sum_parts(qh + 128 + 2 * i, a.np, a.pstride);
        od = sum_parts(qh + 128 + 2 * i + 1, a.np, a.pstride);
        cs = a.cs[(size_t)__shfl(dl.pos, b) * 32 + i];  // b differs between the wave's halves
    }
    __syncthreads();
    // B operand: column n = hi (n < 8) or lo (n >= 8) of sequence n & 7, k = 32 ks + 8 g .. + 7
    v8bf qb[4];
    {
        const int m0 = n < 8 ? -1 : 0, m1 = n < 8 ? 0 : -1;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const v4f x0 = *(const v4f *)&qn8[n & 7][32 * ks + 8 * g];
            const v4f x1 = *(const v4f *)&qn8[n & 7][32 * ks + 8 * g + 4];
            v8bf hi, lo;
            split8_cvt(x0, x1, hi, lo);
            const v4i hv = __builtin_bit_cast(v4i, hi), lv = __builtin_bit_cast(v4i, lo);
            qb[ks] = __builtin_bit_cast(v8bf, (hv & m0) | (lv & m1));
        }
    }
    v4f acc[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
        acc[tt] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) acc[tt] = mfma_bf16(wa[tt][ks], qb[ks], acc[tt]);
    }
    if (qq == 0 && js < nseq) {
        const int i = tid & 31;
        const float ec = ev * cs.x, os = od * cs.y, oc = od * cs.x, es = ev * cs.y;
        float *qrow = a.qf + ((size_t)b * NH + h) * 576;
        qrow[512 + i] = ec - os;
        qrow[544 + i] = oc + es;
    }
    // lanes n < 8: q_lat of sequence n = hi column + lo column (lane n + 8: row_ror:8)
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
        v4f v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = acc[tt][i] + dpp_f32<0x128>(acc[tt][i]);
        if (n < 8 && n < nseq)
            *(v4f *)(a.qf + ((size_t)(8 * g8 + n) * NH + h) * 576 + 128 * qq + 32 * w + 16 * tt + 4 * g) = v;
    }
}

__global__ __launch_bounds__(256) void k_qprep(SeqTable t, Dims d, QprepArgs a) {
    qprep_body(t, d, a, blockIdx.x);
}

// Blocks [0, na) append the new history rows, the rest prepare the queries: the two stages
// read different parts of the same projection and are independent.
__global__ __launch_bounds__(256) void k_append_qprep(SeqTable t, Dims d, AppendArgs aa, QprepArgs qa, int na) {
    if ((int)blockIdx.x < na) append_body(t, d, aa, blockIdx.x);
    else if (qa.quarter) qprep_quarter(t, qa, blockIdx.x - na, d.NH);
    else qprep_body(t, d, qa, blockIdx.x - na);
}

static QprepArgs qprep_args(int fmt, const Dims &d, const uint16_t *kv_b, const uint16_t *ukt,
                            const float2 *rope_cs, const DecodeWork &w, bool quantize) {
    QprepArgs a;
    a.y = w.y;
    a.kv_b = kv_b;
    a.ukt = ukt;
    a.cs = rope_cs;
    a.qf = w.qf;
    a.qhi = w.qhi;
    a.qlo = w.qlo;
    a.qs = w.qs;
    a.qrhi = w.qrhi;
    a.qrlo = w.qrlo;
    a.ldy = d.QO + d.KVO;
    a.np = w.ynp > 1 ? w.ynp : 1;
    a.pstride = w.ypstride;
    a.fmt = fmt;
    a.quantize = quantize ? 1 : 0;
    a.quarter = 0;
    return a;
}

hipError_t launch_qprep(hipStream_t st, int fmt, const SeqTable &t, const Dims &d,
                        const uint16_t *kv_b, const float2 *rope_cs, const DecodeWork &w,
                        bool quantize) {
    if (d.R > kMaxR || d.DN > kMaxDN || d.DR > kMaxDR) return hipErrorInvalidValue;
    const QprepArgs a = qprep_args(fmt, d, kv_b, nullptr, rope_cs, w, quantize);
    hipLaunchKernelGGL(k_qprep, dim3(t.n * d.NH), dim3(256), 0, st, t, d, a);
    return hipGetLastError();
}

hipError_t launch_append_qprep(hipStream_t st, int fmt, const SeqTable &t, const Dims &d,
                               const float *y, int ldy, int koff, int ynp, size_t ypstride,
                               const uint16_t *kv_a_norm, float eps, const float2 *rope_cs,
                               const uint16_t *kv_b, const uint16_t *ukt, const DecodeWork &w, bool quantize) {
    if (d.R > kMaxR || d.DN > kMaxDN || d.DR > kMaxDR || (ynp != 1 && ynp != kGemvKs))
        return hipErrorInvalidValue;
    const AppendArgs aa = append_args(fmt, d, y, ldy, koff, ynp, ypstride, kv_a_norm, eps, rope_cs, w,
                                      false, 0);
    QprepArgs qa = qprep_args(fmt, d, kv_b, ukt, rope_cs, w, quantize);
    // fp32 query rows (no int8 operands): a quarter of the latent columns per block
    qa.quarter = !quantize && fmt != kFmtExp && d.R == 512 && d.DN == 128 && d.DR == 64 && d.QD == 192 &&
                 ukt != nullptr ? 1 : 0;
    const int nq = qa.quarter ? (t.n + 7) / 8 * d.NH * 4 : t.n * d.NH;
    hipLaunchKernelGGL(k_append_qprep, dim3(t.n + nq), dim3(256), 0, st, t, d, aa, qa, t.n);
    return hipGetLastError();
}

// ================================================================ attention ============

struct AttnArgs {
    // Read first by every workgroup (kernel arguments live in device memory and the first read
    // of each 64-byte line is a round trip): the fields the start-up needs come first; the
    // workgroup's SeqDesc comes from the lanes' reads of the table (seq_of) in the same round
    // trip.
    float *part;
    const float *qf;
    const int8_t *qhi, *qlo;
    const float *qs;
    const uint16_t *qrhi, *qrlo;
    float *scores;
    int rps, lmax;
    float smscale;
    int members;  // > 0: a block launch of that many members (seq_of)
    int nseq;     // = t.n
    Dims d;
    SeqTable t;
    FqArgs fq;    // the fused query preparation and append (k_attn_q8_mfma<., true>)
};

// The arguments a workgroup needs before its first loads, passed as leading scalar kernel
// arguments: the leading scalar arguments, up to 14 dwords, are preloaded into SGPRs when the
// wave starts (-amdgpu-kernarg-preload-count=16), so they cost no memory round trip. The order
// puts first what the first loads need (members, nseq, the query operands); part, which only
// the closing stores use, comes last and is read from the argument block.
struct AttnHot {
    float *part;
    const float *qf;
    const int8_t *qhi, *qlo;
    const float *qs;
    const uint16_t *qrhi, *qrlo;
    int members, nseq;  // members: > 0 a block launch (seq_of); a fused Q8 launch: -(its split count)
};
#define KVL_ATTN_HOT_PARAMS                                                                        \
    int members_, int nseq_, const int8_t *qhi_, const int8_t *qlo_, const uint16_t *qrhi_,         \
        const uint16_t *qrlo_, const float *qs_, const float *qf_, float *part_
#define KVL_ATTN_HOT_INIT const AttnHot h{part_, qf_, qhi_, qlo_, qs_, qrhi_, qrlo_, members_, nseq_}

constexpr int kXcds = 8;  // XCDs of an MI355X; workgroups are dispatched to them round-robin

// Block -> (sequence, split): splits of the sequences are numbered consecutively.
__device__ __forceinline__ int find_seq(const SeqTable &t, int bid) {
    int b = 0;
    for (int i = 1; i < t.n; ++i)
        if (bid >= t.s[i].split0) b = i;
    return b;
}

// Workgroup -> (sequence b, split, index of its partial). A normal launch numbers the splits of
// its sequences consecutively. A block launch (members > 0: the sequences are the tokens of one
// block over a shared history, each with the split plan of its lone decode) goes split-major and
// XCD-affine: workgroup i runs on XCD i % kXcds, and split s of every member sits at position
// members * (s / kXcds) + member of XCD s % kXcds's order, so the members of a split run at the
// same time on one XCD and its L2 serves the history rows they share. A workgroup past its
// member's last split has nothing to do (false).
// Sequence b's descriptor comes from desc_lane / desc_pick, b from a ballot over the lanes'
// split0 (a lone decode's attention launch: 12.5 -> 10.3 us at 8K Q8 rows, 18.3 -> 16.5 us at
// 32K against indexing the table by b once b is known).
// XL (the Q8 launch that also combines, nseq a multiple of kXcds, every sequence with the same
// split count ns, its splits consecutive): sequence-major per XCD, workgroup i takes sequence
// i % kXcds + kXcds * ((i / kXcds) / ns), split (i / kXcds) % ns, so that all splits of a sequence
// run on one XCD and its partials stay in that XCD's L2 for the combine (q8_comb_tail).
template <bool XL = false>
__device__ __forceinline__ bool seq_of(const AttnArgs &a, const AttnHot &h, int &b, int &split, int &pidx, SeqDesc &s) {
    const int sid = blockIdx.x, lane = threadIdx.x & 63;
    const DescLane m = desc_lane(a.t);
    if constexpr (XL) {
        const int ns = lane_pick(m.nsplit, 0), j = sid / kXcds;
        b = sid % kXcds + kXcds * (j / ns);
        split = j % ns;
        s = desc_pick(m, b);
        pidx = s.split0 + split;
        return true;
    }
    if (h.members > 0) {
        const int j = sid / kXcds;
        b = j % h.members;
        split = kXcds * (j / h.members) + sid % kXcds;
    } else {
        b = __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane >= 1 && lane < h.nseq && sid >= m.split0));
        split = sid - lane_pick(m.split0, b);
    }
    s = desc_pick(m, b);
    if (h.members > 0) {
        if (split >= s.nsplit) return false;
        pidx = s.split0 + split;
    } else {
        pidx = sid;
    }
    return true;
}

// ---- generic VALU path: any dims and formats, one block per problem -----------------
// Problem = one sequence (compressed: all NH heads share the rows) or one (sequence, head)
// (expanded). Two-pass softmax over the full history; partial written with one split.
template <int FMT>
__device__ __forceinline__ float score_elem(const SeqDesc &s, const Dims &d, int h, int j, int k) {
    if (FMT == kFmtQ8) {
        if (k < d.R) return (float)((const int8_t *)s.a)[(size_t)j * d.R + k] * ((const float *)s.b)[j];
        return bf16_to_f32(((const uint16_t *)s.c)[(size_t)j * d.DR + (k - d.R)]);
    } else if (FMT == kFmtF32) {
        if (k < d.R) return ((const float *)s.a)[(size_t)j * d.R + k];
        return ((const float *)s.b)[(size_t)j * d.DR + (k - d.R)];
    } else if (FMT == kFmtBF16) {
        if (k < d.R) return bf16_to_f32(((const uint16_t *)s.a)[(size_t)j * d.R + k]);
        return bf16_to_f32(((const uint16_t *)s.b)[(size_t)j * d.DR + (k - d.R)]);
    } else {
        return ((const float *)s.a)[((size_t)j * d.NH + h) * d.QD + k];
    }
}
template <int FMT>
__device__ __forceinline__ float value_elem(const SeqDesc &s, const Dims &d, int h, int j, int k) {
    if (FMT == kFmtQ8) return (float)((const int8_t *)s.a)[(size_t)j * d.R + k] * ((const float *)s.b)[j];
    if (FMT == kFmtF32) return ((const float *)s.a)[(size_t)j * d.R + k];
    if (FMT == kFmtBF16) return bf16_to_f32(((const uint16_t *)s.a)[(size_t)j * d.R + k]);
    return ((const float *)s.b)[((size_t)j * d.NH + h) * d.DV + k];
}

template <int FMT>
__global__ __launch_bounds__(256) void k_attn_generic(AttnArgs a) {
    __shared__ float red[256];
    __shared__ float ml[2 * 64];
    const Dims &d = a.d;
    const int p = blockIdx.x, tid = threadIdx.x;
    const bool exp = FMT == kFmtExp;
    const int b = exp ? p / d.NH : p, h0 = exp ? p % d.NH : 0;
    const int G = exp ? 1 : d.NH, DS = exp ? d.QD : d.R + d.DR, DVm = exp ? d.DV : d.R;
    const SeqDesc &s = a.t.s[b];
    const int L = s.len;
    const float *q = a.qf + ((size_t)b * d.NH + h0) * DS;
    float *sc = a.scores + (size_t)p * G * a.lmax;
    for (int idx = tid; idx < G * L; idx += 256) {
        const int g = idx / L, j = idx % L;
        float acc = 0.f;
        for (int k = 0; k < DS; ++k) acc = fmaf(q[(size_t)g * DS + k], score_elem<FMT>(s, d, h0 + g, j, k), acc);
        sc[(size_t)g * a.lmax + j] = acc * a.smscale;
    }
    __syncthreads();
    for (int g = 0; g < G; ++g) {
        float m = -INFINITY;
        for (int j = tid; j < L; j += 256) m = fmaxf(m, sc[(size_t)g * a.lmax + j]);
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
            const float e = __expf(sc[(size_t)g * a.lmax + j] - m);
            sc[(size_t)g * a.lmax + j] = e;
            sum += e;
        }
        red[tid] = sum;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if (tid < o) red[tid] += red[tid + o];
            __syncthreads();
        }
        if (tid == 0) {
            ml[2 * g] = m;
            ml[2 * g + 1] = red[0];
        }
        __syncthreads();
    }
    const int split = exp ? p : s.split0;
    float *P = a.part + (size_t)split * G * (DVm + 2);
    for (int idx = tid; idx < G * DVm; idx += 256) {
        const int g = idx / DVm, k = idx % DVm;
        float acc = 0.f;
        for (int j = 0; j < L; ++j) acc = fmaf(sc[(size_t)g * a.lmax + j], value_elem<FMT>(s, d, h0 + g, j, k), acc);
        P[idx] = acc;
    }
    for (int g = tid; g < G; g += 256) {
        P[(size_t)G * DVm + g] = ml[2 * g];
        P[(size_t)G * DVm + G + g] = ml[2 * g + 1];
    }
}

// s_waitcnt vmcnt(n) for the counts the DMA pipelines of the attention kernels use (n
// wave-uniform; any other n waits for everything).
__device__ __forceinline__ void wait_vm(int n) {
    switch (n) {
    case 0: wait_vmcnt<0>(); break;
    case 2: wait_vmcnt<2>(); break;
    case 3: wait_vmcnt<3>(); break;
    case 8: wait_vmcnt<8>(); break;
    case 9: wait_vmcnt<9>(); break;
    case 10: wait_vmcnt<10>(); break;
    case 11: wait_vmcnt<11>(); break;
    case 16: wait_vmcnt<16>(); break;
    case 18: wait_vmcnt<18>(); break;
    case 19: wait_vmcnt<19>(); break;
    default: wait_vmcnt<0>(); break;
    }
}

// ---- bf16 MFMA path (BF16 history, NH=16, R=512, DR=64) -------------------------------
// Two workgroups of four waves per CU (two waves per SIMD, so that one workgroup's softmax, LDS
// round trips and DMA waits overlap the other's MFMAs) each stream a split-K slice in chunks of
// 32 rows (36 KB: 32 KB of latents, 4 KB of RoPE keys) through a ring of two LDS slots filled by
// global_load_lds_dwordx4: chunk k is computed while chunk k+1 lands. The rows are exact bf16
// MFMA operands, so only the query side and the softmax weights are split:
//   scores: M = 16 heads, N = 16 rows, K = 576. Wave w takes rows 16 (w & 1) .. +15 and the
//     k-blocks 9 (w >> 1) .. +8 of 32 against the bf16 hi | lo split of q * softmax scale (two
//     v_mfma_f32_16x16x32_bf16 per block); the two k-halves are summed through LDS;
//   softmax: every wave keeps the online statistics of all 16 heads (the same arithmetic in
//     each wave); lane group g takes chunk rows 8g .. 8g+7; the reference max moves lazily (p <= 4);
//   mix: wave w owns latent columns 128w .. +127 (M = heads, N = 16 columns, K = the 32 rows),
//     p split into bf16 hi | lo, the rows read transposed by ds_read_b64_tr_b16, fp32
//     accumulators rescaled by exp(m_old - m_new) when the reference max moves.
// The 16-byte slots of a latent row are XOR-swizzled by b16_swz(row), so that the score reads
// (16 rows, one slot) and the transposed reads (4 rows x 32 bytes per 16 lanes, 8 rows per half
// wave) spread over the LDS banks.
constexpr int kB16Ch = 32;
constexpr int kB16Ring = 2;
constexpr int kB16LatB = kB16Ch * 1024;            // latents of a chunk
constexpr int kB16Slot = kB16LatB + kB16Ch * 128;  // + RoPE keys
constexpr int kB16SpHs = 36;                       // floats per head in a score half: 32 + 4
constexpr int kB16SpOff = kB16Ring * kB16Slot;     // score halves [2][16 heads][kB16SpHs]
constexpr int kB16SmemB = kB16SpOff + 2 * 16 * kB16SpHs * 4;
static_assert(kB16SmemB <= 160 * 1024, "LDS of one CU");

// bits (r3, r2, r1, r0) of a chunk row -> slot XOR (r3, r1, r0, r2): a bijection on 16 rows, and
// (r3, r1, r0) -> distinct slot pairs for the 8 rows of a transposed half-wave read
__device__ __forceinline__ int b16_swz(int row) { return ((row & 3) << 1) | ((row >> 2) & 1) | (row & 8); }

// Max / sum over lanes l, l ^ 16, l ^ 32, l ^ 48 with the gfx950 lane-swap instructions (VALU,
// no LDS round trip): v_permlane16_swap with both operands v gives every lane the values of its
// lane pair (l & ~16, l | 16), v_permlane32_swap those of (l & ~32, l | 32); the lower lane's value
// comes first, so every lane computes the same result.
__device__ __forceinline__ float xgroup_max(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
__device__ __forceinline__ float xgroup_sum(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

constexpr float kB16LnPmax = 1.3862944f;  // ln 4: the weights p_j = exp(s_j - m) stay <= 4

typedef short v4s __attribute__((ext_vector_type(4)));
// ds_read_b64_tr_b16: within each 16-lane group, destination lane i element e is element i & 3
// of the four addressed by source lane 4e + (i >> 2).
__device__ __forceinline__ v4s lds_read_tr16(const uint8_t *p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)(p));
}

template <bool ONCE>  // ONCE: each history row is read by one workgroup (non-temporal loads)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_attn_bf16_mfma(KVL_ATTN_HOT_PARAMS, AttnArgs a) {
    KVL_ATTN_HOT_INIT;
    __shared__ __attribute__((aligned(16))) uint8_t smem[kB16SmemB];
    const int tid = threadIdx.x, l = tid & 63, n = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int b, split, pidx;
    SeqDesc s;
    if (!seq_of(a, h, b, split, pidx, s)) return;
    const int r0 = split * s.rps;
    const int r1 = split == s.nsplit - 1 ? s.len : r0 + s.rps;  // last split takes the rest
    const int nch = (r1 - r0 + kB16Ch - 1) / kB16Ch;
    const uint16_t *glat = (const uint16_t *)s.a;
    const uint16_t *grope = (const uint16_t *)s.b;
    constexpr bool once = ONCE;
    const uint32_t sbase = lds_addr(smem);
    float *sp = (float *)(smem + kB16SpOff);
    const int rb = w & 1, kh = w >> 1;

    // DMA per chunk and wave: latent rows 8w .. 8w+7, one 1 KB instruction per row (lane i
    // writes physical slot i, which holds logical slot i ^ b16_swz(row)); RoPE rows 8w .. 8w+7,
    // one instruction (lane i: row 8w + (i >> 3), physical slot i & 7 = logical (i & 7) ^
    // (row & 7)). Rows past the split end (last chunk only) re-read the split's last row (in
    // bounds); their scores are masked.
    auto issue = [&](int c) __attribute__((always_inline)) {
        const uint32_t buf = sbase + (uint32_t)((c % kB16Ring) * kB16Slot);
        const int rbase = r0 + c * kB16Ch;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int row = 8 * w + k;
            const int gr = min(rbase + row, r1 - 1);
            dma_hist_b128(glat + (size_t)gr * 512 + 8 * (l ^ b16_swz(row)), buf + (uint32_t)(row * 1024), once);
        }
        const int row = 8 * w + (l >> 3);
        const int gr = min(rbase + row, r1 - 1);
        dma_hist_b128(grope + (size_t)gr * 64 + 8 * ((l & 7) ^ (row & 7)), buf + (uint32_t)(kB16LatB + w * 1024), once);
    };

    // query operands (A of the score MFMAs: head n, k = 32 kb + 8g .. +7). Chunk 0's DMA goes out
    // first; the query loads follow it.
    v8bf qh[9], ql[9];
    issue(0);
    {
        const float *qrow = h.qf + ((size_t)b * 16 + n) * 576 + 8 * g + 32 * 9 * kh;
        v4f qv[18];
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            qv[2 * j] = *(const v4f *)(qrow + 32 * j);
            qv[2 * j + 1] = *(const v4f *)(qrow + 32 * j + 4);
        }
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            split8_cvt(qv[2 * j] * a.smscale, qv[2 * j + 1] * a.smscale, qh[j], ql[j]);
        }
    }

    // score operand offsets (row srow of the chunk, slot 4 kb + g of its latents / RoPE key)
    const int srow = 16 * rb + n;
    int bofs[9];
#pragma unroll
    for (int j = 0; j < 9; ++j) {
        const int kb = 9 * kh + j;
        bofs[j] = kb < 16 ? srow * 1024 + 16 * ((4 * kb + g) ^ b16_swz(srow))
                          : kB16LatB + srow * 128 + 16 * ((4 * (kb - 16) + g) ^ (srow & 7));
    }
    // transposed reads of column block 8w + t: half h covers rows 8g + 4h .. +3 (lane n
    // addresses row 8g + 4h + (n >> 2), columns 4 (n & 3) .. +3 of the block)
    int tro[2][8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int row = 8 * g + 4 * h + (n >> 2);
#pragma unroll
        for (int t = 0; t < 8; ++t)
            tro[h][t] = row * 1024 + 16 * ((2 * (8 * w + t) + ((n >> 1) & 1)) ^ b16_swz(row)) + 8 * (n & 1);
    }

    float m_run = -INFINITY, l_run = 0.f;  // head n
    v4f acc[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < nch; ++k) {
        // this wave's DMA of chunk k has landed (the only one in flight)
        wait_vm(0);
        lds_barrier();  // chunk k complete; every wave is done with chunk k-1's slot and the scores
        if (k + 1 < nch) issue(k + 1);
        const uint8_t *buf = smem + (k % kB16Ring) * kB16Slot;
        v4f dp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            const v8bf bv = *(const v8bf *)(buf + bofs[j]);
            dp = mfma_bf16(qh[j], bv, dp);
            dp = mfma_bf16(ql[j], bv, dp);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sp[(kh * 16 + 4 * g + i) * kB16SpHs + srow] = dp[i];
        lds_barrier();  // both k-halves of every score are in LDS
        const float *s0 = sp + n * kB16SpHs + 8 * g, *s1 = sp + (16 + n) * kB16SpHs + 8 * g;
        const v4f a0 = *(const v4f *)s0, a1 = *(const v4f *)(s0 + 4);
        const v4f c0 = *(const v4f *)s1, c1 = *(const v4f *)(s1 + 4);
        const int nv = r1 - (r0 + k * kB16Ch);  // valid rows of the chunk (>= 1)
        float sc[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sc[e] = 8 * g + e < nv ? a0[e] + c0[e] : -INFINITY;
            sc[e + 4] = 8 * g + e + 4 < nv ? a1[e] + c1[e] : -INFINITY;
        }
        const float cmax = xgroup_max(
            fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7]))));
        // lazy reference max: it moves only when the chunk exceeds it by more than ln 4 (every
        // head in the first chunk, where it is -inf); then the accumulators of the heads concerned
        // are rescaled by alpha = exp(m_old - m_new) (0 from -inf). All four waves hold the same
        // statistics, so they take the same branch.
        const bool mv = cmax > m_run + kB16LnPmax;
        if (__any(mv)) {
            const float mnew = mv ? cmax : m_run;
            const float alpha = mv ? __expf(m_run - mnew) : 1.0f;
            m_run = mnew;
            l_run *= alpha;
            float ad[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) ad[i] = __shfl(alpha, 4 * g + i);
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[t][i] *= ad[i];
        }
        float p[8], psum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            p[e] = __expf(sc[e] - m_run);
            psum += p[e];
        }
        l_run += xgroup_sum(psum);
        v8bf ph, pl;
        split8_cvt(v4f{p[0], p[1], p[2], p[3]}, v4f{p[4], p[5], p[6], p[7]}, ph, pl);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const v4s lo4 = lds_read_tr16(buf + tro[0][t]);
            const v4s hi4 = lds_read_tr16(buf + tro[1][t]);
            const v8bf bt = __builtin_bit_cast(v8bf, __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
            acc[t] = mfma_bf16(ph, bt, acc[t]);
            acc[t] = mfma_bf16(pl, bt, acc[t]);
        }
    }
    float *P = h.part + (size_t)pidx * 16 * 514;
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) P[(4 * g + i) * 512 + 128 * w + 16 * t + n] = acc[t][i];
    if (w == 0 && g == 0) {
        P[8192 + n] = m_run;
        P[8192 + 16 + n] = l_run;
    }
}

// ---- FP32 history on bf16 MFMA (NH=16, R=512, DR=64) ----------------------------------
// The BF16 kernel's pipeline over FP32 rows: a chunk is 16 rows (36 KB: 32 KB of latents, 4 KB
// of RoPE keys, the size of a BF16 chunk), streamed by DMA into a ring of two LDS slots (chunk
// k computed while chunk k+1 lands); two workgroups run on each CU (two waves per SIMD), so that
// one workgroup's conversion, softmax and DMA waits overlap the other's MFMAs.
// Each fp32 row becomes two bf16 "virtual rows", hi = bf16(x) and lo = bf16(x - hi) (x - hi is
// exact, |x - hi - lo| <= 2^-18 |x|): virtual rows 0-15 are the hi parts of rows 0-15, 16-31 their
// lo parts, laid out as a 32-row BF16 chunk. Wave w loads rows 4w .. 4w+3 so that their fp32
// bytes land exactly where their virtual rows go (latent columns 0-255 of row r in virtual row
// r's kilobyte, 256-511 in virtual row 16 + r's; the four RoPE rows in the wave's quarter of the
// RoPE area) and converts them in place once its own DMA has landed, before the step barrier:
// no extra barrier, no extra LDS. The BF16 kernel's score, softmax and mix then run on the 32
// virtual rows: a row's score is the sum of its two virtual rows' scores (q hi + lo against
// row hi + lo: all four products), and both virtual rows of a row carry its weight p (hi + lo),
// so the mix adds p (hi + lo) of the row. Per history byte this is the BF16 kernel's MFMA work.
// RoPE quarter of wave w (1 KB at kB16LatB + w * 1024): local virtual row k = 0..3 the hi parts,
// 4..7 the lo parts of rows 4w + (k & 3), 128 bytes each, 16-byte slot s at s ^ f32r_swz(row)
// (row = the row in the chunk) so that the score reads of 8 rows fall in distinct banks.
constexpr int kF32Ch = 16;
constexpr int kF32Ring = 2;
constexpr int kF32SpOff = kF32Ring * kB16Slot;
constexpr int kF32SmemB = kF32SpOff + 2 * 16 * kB16SpHs * 4;
typedef int v2i __attribute__((ext_vector_type(2)));
__device__ __forceinline__ int f32r_swz(int row) { return (row >> 1) & 7; }

template <bool ONCE>  // ONCE: each history row is read by one workgroup (non-temporal loads)
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_attn_f32_mfma(KVL_ATTN_HOT_PARAMS, AttnArgs a) {
    KVL_ATTN_HOT_INIT;
    __shared__ __attribute__((aligned(16))) uint8_t smem[kF32SmemB];
    const int tid = threadIdx.x, l = tid & 63, n = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int b, split, pidx;
    SeqDesc s;
    if (!seq_of(a, h, b, split, pidx, s)) return;
    const int r0 = split * s.rps;
    const int r1 = split == s.nsplit - 1 ? s.len : r0 + s.rps;  // last split takes the rest
    const int nch = (r1 - r0 + kF32Ch - 1) / kF32Ch;
    const float *glat = (const float *)s.a;
    const float *grope = (const float *)s.b;
    constexpr bool once = ONCE;
    const uint32_t sbase = lds_addr(smem);
    float *sp = (float *)(smem + kF32SpOff);
    const int rb = w & 1, kh = w >> 1;

    // DMA per chunk and wave: rows 4w .. 4w+3, two 1 KB instructions per row (latent columns
    // 0-255 -> virtual row r, 256-511 -> virtual row 16 + r), one for the four RoPE rows (lane i:
    // row 4w + (i >> 4), columns 4 (i & 15) .. +3). Rows past the split end (last chunk only)
    // re-read the split's last row (in bounds); their scores are masked.
    auto issue = [&](int c) __attribute__((always_inline)) {
        const uint32_t buf = sbase + (uint32_t)((c % kF32Ring) * kB16Slot);
        const int rbase = r0 + c * kF32Ch;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 4 * w + i;
            const int gr = min(rbase + row, r1 - 1);
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
                dma_hist_b128(glat + (size_t)gr * 512 + 256 * hf + 4 * l, buf + (uint32_t)((16 * hf + row) * 1024),
                              once);
        }
        const int row = 4 * w + (l >> 4);
        const int gr = min(rbase + row, r1 - 1);
        dma_hist_b128(grope + (size_t)gr * 64 + 4 * (l & 15), buf + (uint32_t)(kB16LatB + w * 1024), once);
    };
    // In-place conversion of this wave's rows of chunk c (its DMA has landed): every lane reads
    // its fp32 values first, then writes the hi and lo words (the wave's bytes only).
    auto convert = [&](int c) __attribute__((always_inline)) {
        uint8_t *buf = smem + (c % kF32Ring) * kB16Slot;
        v4f x[4][2];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 4 * w + i;  // columns 8l .. 8l+7: lanes 0-31 in row's kilobyte, 32-63 in 16 + row's
            const uint8_t *src = buf + (l < 32 ? row * 1024 + 32 * l : (16 + row) * 1024 + 32 * (l - 32));
            x[i][0] = *(const v4f *)src;
            x[i][1] = *(const v4f *)(src + 16);
        }
        uint8_t *rq = buf + kB16LatB + w * 1024;
        const v4f xr = *(const v4f *)(rq + 16 * l);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 4 * w + i;
            v8bf hi, lo;
            split8_cvt(x[i][0], x[i][1], hi, lo);
            const int slot = 16 * (l ^ b16_swz(row));
            *(v8bf *)(buf + row * 1024 + slot) = hi;
            *(v8bf *)(buf + (16 + row) * 1024 + slot) = lo;
        }
        {
            const int k = l >> 4, row = 4 * w + k;
            v8bf hi, lo;
            split8_cvt(xr, v4f{0.f, 0.f, 0.f, 0.f}, hi, lo);
            const int o = 16 * (((l & 15) >> 1) ^ f32r_swz(row)) + 8 * (l & 1);
            const v4i hv = __builtin_bit_cast(v4i, hi), lv = __builtin_bit_cast(v4i, lo);
            *(v2i *)(rq + k * 128 + o) = v2i{hv.x, hv.y};
            *(v2i *)(rq + (4 + k) * 128 + o) = v2i{lv.x, lv.y};
        }
    };

    // query operands (A of the score MFMAs: head n, k = 32 kb + 8g .. +7), as the BF16 kernel
    v8bf qh[9], ql[9];
    issue(0);
    {
        const float *qrow = h.qf + ((size_t)b * 16 + n) * 576 + 8 * g + 32 * 9 * kh;
        v4f qv[18];
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            qv[2 * j] = *(const v4f *)(qrow + 32 * j);
            qv[2 * j + 1] = *(const v4f *)(qrow + 32 * j + 4);
        }
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            split8_cvt(qv[2 * j] * a.smscale, qv[2 * j + 1] * a.smscale, qh[j], ql[j]);
        }
    }

    // score operand offsets: virtual row srow = 16 rb + n (row n's hi part for rb = 0, lo for 1)
    const int srow = 16 * rb + n;
    int bofs[9];
#pragma unroll
    for (int j = 0; j < 9; ++j) {
        const int kb = 9 * kh + j;
        bofs[j] = kb < 16 ? srow * 1024 + 16 * ((4 * kb + g) ^ b16_swz(srow))
                          : kB16LatB + (n >> 2) * 1024 + ((n & 3) + 4 * rb) * 128 +
                                16 * ((4 * (kb - 16) + g) ^ f32r_swz(n));
    }
    // transposed reads of column block 8w + t over the 32 virtual rows (as the BF16 kernel)
    int tro[2][8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int row = 8 * g + 4 * h + (n >> 2);
#pragma unroll
        for (int t = 0; t < 8; ++t)
            tro[h][t] = row * 1024 + 16 * ((2 * (8 * w + t) + ((n >> 1) & 1)) ^ b16_swz(row)) + 8 * (n & 1);
    }

    float m_run = -INFINITY, l_run = 0.f;  // head n
    v4f acc[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
    const int rg = 8 * (g & 1);  // the rows whose softmax weights lane group g holds
    for (int k = 0; k < nch; ++k) {
        // this wave's DMA of chunk k has landed (the only one in flight)
        wait_vm(0);
        convert(k);
        lds_barrier();  // chunk k converted; every wave is done with chunk k-1's slot and the scores
        if (k + 1 < nch) issue(k + 1);
        const uint8_t *buf = smem + (k % kF32Ring) * kB16Slot;
        v4f dp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 9; ++j) {
            const v8bf bv = *(const v8bf *)(buf + bofs[j]);
            dp = mfma_bf16(qh[j], bv, dp);
            dp = mfma_bf16(ql[j], bv, dp);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sp[(kh * 16 + 4 * g + i) * kB16SpHs + srow] = dp[i];
        lds_barrier();  // both k-halves of every virtual row's score are in LDS
        // row rg + e: (hi, first k-half + second) + (lo, first + second)
        const float *s0 = sp + n * kB16SpHs + rg, *s1 = sp + (16 + n) * kB16SpHs + rg;
        const v4f a0 = *(const v4f *)s0, a1 = *(const v4f *)(s0 + 4);
        const v4f c0 = *(const v4f *)s1, c1 = *(const v4f *)(s1 + 4);
        const v4f a2 = *(const v4f *)(s0 + 16), a3 = *(const v4f *)(s0 + 20);
        const v4f c2 = *(const v4f *)(s1 + 16), c3 = *(const v4f *)(s1 + 20);
        const int nv = r1 - (r0 + k * kF32Ch);  // valid rows of the chunk (>= 1)
        float sc[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            sc[e] = rg + e < nv ? (a0[e] + c0[e]) + (a2[e] + c2[e]) : -INFINITY;
            sc[e + 4] = rg + e + 4 < nv ? (a1[e] + c1[e]) + (a3[e] + c3[e]) : -INFINITY;
        }
        const float cmax = xgroup_max(
            fmaxf(fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])), fmaxf(fmaxf(sc[4], sc[5]), fmaxf(sc[6], sc[7]))));
        // lazy reference max, as the BF16 kernel (all four waves hold the same statistics)
        const bool mv = cmax > m_run + kB16LnPmax;
        if (__any(mv)) {
            const float mnew = mv ? cmax : m_run;
            const float alpha = mv ? __expf(m_run - mnew) : 1.0f;
            m_run = mnew;
            l_run *= alpha;
            float ad[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) ad[i] = __shfl(alpha, 4 * g + i);
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[t][i] *= ad[i];
        }
        float p[8], psum = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            p[e] = __expf(sc[e] - m_run);
            psum += p[e];
        }
        // lane groups g and g ^ 2 hold the same rows (hi and lo virtual rows): count them once
        l_run += xgroup_sum(g < 2 ? psum : 0.f);
        v8bf ph, pl;
        split8_cvt(v4f{p[0], p[1], p[2], p[3]}, v4f{p[4], p[5], p[6], p[7]}, ph, pl);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const v4s lo4 = lds_read_tr16(buf + tro[0][t]);
            const v4s hi4 = lds_read_tr16(buf + tro[1][t]);
            const v8bf bt = __builtin_bit_cast(v8bf, __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
            acc[t] = mfma_bf16(ph, bt, acc[t]);
            acc[t] = mfma_bf16(pl, bt, acc[t]);
        }
    }
    float *P = h.part + (size_t)pidx * 16 * 514;
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) P[(4 * g + i) * 512 + 128 * w + 16 * t + n] = acc[t][i];
    if (w == 0 && g == 0) {
        P[8192 + n] = m_run;
        P[8192 + 16 + n] = l_run;
    }
}

// ---- int8 MFMA path (Q8 history, NH=16, R=512, DR=64) ---------------------------------
// One workgroup of 8 waves (two per SIMD) per CU streams its split-K slice in chunks of 64
// rows. The waves specialise, and the two roles run one chunk apart:
//   score waves 0-3 (rows 16w .. 16w+15 of a chunk) take chunk k in step k: scores, softmax,
//     and the quantised mix weights of their rows into LDS;
//   mix waves 4-7 (latent columns 128(w-4) .. +127) take chunk k-1 in step k: they issue the
//     history DMA (global_load_lds_dwordx4 into a ring of four 32 KB code slots: chunk k-1
//     being mixed, chunk k being scored, chunks k+1 and k+2 in flight) and accumulate the mix.
// A score wave's softmax and quantisation (VALU) thus overlap the mix wave's MFMAs and DMA on
// the same SIMD. One barrier per step orders everything in the common case: the weights of
// chunk k are written before it and read after it, the mix waves have waited for chunk k+1's
// DMA and finished reading chunk k-1's slot before it.
// Scores: v_mfma_i32_16x16x64_i8 on the raw int8 codes against the int8 hi/lo split of q_lat
// (exact integer dot products), plus bf16 MFMA on the bf16 RoPE keys (loaded by the score
// waves straight into registers, one chunk ahead) against the hi/lo bf16 split of q_rope. The
// row scale factors out of the dot (score_j = s_j * q_lat . c_j + q_rope . k_j).
// Mix: the weights p_j*s_j (p_j <= kQ8Pmax against the lazily moved reference max below,
// s_j <= the split's largest scale) are quantised to three int8 levels hi + lo/254 + lo2/254^2
// against kQ8Pmax * that scale (23 bits below the bound: a row whose scale is far below the
// split's largest -- an all-zero latent stored with scale 1, or a flat row beside a
// one-hot-like one -- keeps the precision of its own weight); ds_read_b64_tr_b8 reads the codes
// transposed (16 rows of one column per lane), and v_mfma_i32_16x16x64_i8 accumulates the exact
// integer mix of each level across chunks. A head's reference max only moves when a chunk
// exceeds it by more than ln kQ8Pmax (so p_j <= kQ8Pmax): the score waves then exchange their
// chunk maxima (two more barriers, taken by all eight waves on the same LDS flags), requantise
// the chunk's weights and publish alpha = exp(m_old - m_new); the mix waves rescale their
// accumulators by alpha (in double, each level's rounding remainder carried into the next)
// before they add that chunk. kQ8Pmax = 4 makes these exchanges rare after the first chunk.
constexpr int kQ8Ch = 64;
constexpr float kQ8Pmax = 4.0f;            // bound of p_j = exp(s_j - reference max)
constexpr float kQ8LnPmax = 1.3862944f;    // ln kQ8Pmax
constexpr int kQ8Ring = 4;                          // code slots (chunks k .. k+3)
constexpr int kQ8CodeB = kQ8Ch * 512;               // codes of a chunk
constexpr int kQ8RRing = 3;                         // RoPE-key + scale slots (chunks k .. k+2)
constexpr int kQ8RopeB = kQ8Ch * 128;               // bf16 RoPE keys of a chunk
constexpr int kQ8RSlot = kQ8RopeB + kQ8Ch * 4;      // + the chunk's row scales
constexpr int kQ8RopeOff = kQ8Ring * kQ8CodeB;
constexpr int kQ8Ws = 64;                           // LDS bytes per quantised-weight row
constexpr int kQ8WqB = 3 * 16 * kQ8Ws;              // quantised weights of a chunk (hi, lo, lo2)
constexpr int kQ8WqOff = kQ8RopeOff + kQ8RRing * kQ8RSlot;  // two weight buffers, by chunk parity
constexpr int kQ8FlagOff = kQ8WqOff + 2 * kQ8WqB;   // [2][4] int: a row exceeds the reference max
constexpr int kQ8MlOff = kQ8FlagOff + 2 * 4 * 4;    // [2][4 waves][16] chunk maxima
constexpr int kQ8AlOff = kQ8MlOff + 2 * 4 * 16 * 4; // [2][16] alpha of a moved reference max
constexpr int kQ8LsOff = kQ8AlOff + 2 * 16 * 4;     // [4 waves][16] softmax denominators
constexpr int kQ8SmOff = kQ8LsOff + 4 * 16 * 4;     // [4] largest row scale per score wave
constexpr int kQ8SmemB = kQ8SmOff + 4 * 4;
static_assert(kQ8SmemB <= 160 * 1024, "LDS of one CU");

// ---- query preparation and row append inside the Q8 attention launch ----------------------
// The Kimi-shape decode with the q_proj | kv_a partials of k_gemv_ksplit: instead of a launch of
// its own (k_append_qprep), the work is done by the attention's lowest-numbered workgroups ahead
// of their own split: block i < 16 B prepares the query of (sequence i / 16, head i % 16), block
// 16 B + b appends sequence b's row, with all 512 threads and the arithmetic of qprep_body /
// append_body (so the query operands and the rows are bit-identical to theirs). The results are
// written with device-scope (sc1) stores, which reach memory without a write-back of the L2, and
// counted on per-sequence flags with device-scope atomics; a workgroup's score waves wait for the
// 16 heads of its sequence before they load its query, and the split that holds the new row waits
// for its append before that row's chunk is requested. Workgroups are dispatched in index order,
// so the producers have started whenever anything waits on them; the waits are bounded anyway
// (a timeout raises FqArgs::err and the launch ends with wrong values instead of hanging).

__device__ __forceinline__ void st_sc1_b32(void *p, uint32_t v) {
    asm volatile("global_store_dword %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void st_sc1_b16(void *p, uint32_t v) {
    asm volatile("global_store_short %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ float ld_sc1_f32(const float *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Flag words 128 bytes apart (one line each: the polls of one sequence do not queue behind
// another's at the memory side): query heads of sequence b at kFqFlagStride * b, its row at
// kFqFlagStride * (kMaxBatch + b).
__device__ __forceinline__ unsigned *fq_qflag(const FqArgs &f, int b) { return f.flags + (size_t)kFqFlagStride * b; }
__device__ __forceinline__ unsigned *fq_aflag(const FqArgs &f, int b) {
    return f.flags + (size_t)kFqFlagStride * (kMaxBatch + b);
}

// Lane 0 of the calling wave polls *flag until it reaches target (bounded); the wave's later
// loads are issued after the poll has returned.
__device__ __forceinline__ void fq_wait(const FqArgs &f, const unsigned *flag, unsigned target) {
    if ((threadIdx.x & 63) == 0) {
        const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
        while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
            if (__builtin_amdgcn_s_memrealtime() - t0 > (uint64_t)f.spin) {
                __hip_atomic_store(f.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
    }
}

// Max / double sum over the eight waves of a 512-thread workgroup (waves without values pass
// 0, the neutral element of both: the results equal block256_max / block256_sum_f64 over the
// first four waves bit for bit). red8: 8 entries.
__device__ __forceinline__ float block512_max(float v, float *red8) {
    v = wave_max(v);
    if ((threadIdx.x & 63) == 0) red8[threadIdx.x >> 6] = v;
    __syncthreads();
    return fmaxf(fmaxf(fmaxf(red8[0], red8[1]), fmaxf(red8[2], red8[3])),
                 fmaxf(fmaxf(red8[4], red8[5]), fmaxf(red8[6], red8[7])));
}
__device__ __forceinline__ double block512_sum_f64(double v, double *red8) {
    v = wave_sum_f64(v);
    if ((threadIdx.x & 63) == 0) red8[threadIdx.x >> 6] = v;
    __syncthreads();
    return ((red8[0] + red8[1]) + (red8[2] + red8[3])) + ((red8[4] + red8[5]) + (red8[6] + red8[7]));
}

// Projection counts (kFqFlagLines): line 3 kMaxBatch + i, i < 16 the q rows of head i, i = 16
// the kv_a rows.
__device__ __forceinline__ unsigned *fq_gflag(const FqArgs &f, int i) {
    return f.flags + (size_t)kFqFlagStride * (3 * kMaxBatch + i);
}
// Thread 0 polls *flag until it reaches target (bounded, as fq_wait), then the whole workgroup
// goes on.
__device__ __forceinline__ void fq_wait_all(const FqArgs &f, const unsigned *flag, unsigned target) {
    if (threadIdx.x == 0) {
        const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
        while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
            if (__builtin_amdgcn_s_memrealtime() - t0 > (uint64_t)f.spin) {
                __hip_atomic_store(f.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
    }
    __syncthreads();
}

// The projection's operand normalised in place (FqArgs::xnorm): wave w forms the RMS factor of
// sequence w over its 2048 columns, adding k_rmsnorm's values in k_rmsnorm's order (the sums of its
// threads l, l + 64, l + 128, l + 192, their tree, then the lanes), and every lane scales its own
// columns, so the operand equals that kernel's output bit for bit. Every workgroup reads all of x (64
// KB, from its XCD's L2) beside its 64 KB of weights. Decode stack (27 layers, 8 x 32K rows): the
// launch grows by 2 us and the norm's launch goes, 1539 -> 1513 us. An instance of its own of the
// kCombXcd form: a branch in the others cost the lone decode 0.2 us of 29.3. inv: 8 floats of LDS.
__device__ __forceinline__ void fq_norm_x(const FqArgs &f, int B, int kq, v4f (&xa)[2], v4f (&xb)[2], float *inv) {
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
    const float *xr = f.x + (size_t)min(w, B - 1) * f.ldx;
    float v[4][8];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 8; ++i) v[q][i] = xr[l + 64 * q + 256 * i];
    v4i wt[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) wt[j] = *(const v4i *)(f.xnorm + kq * 512 + (w + 8 * j) * 32 + g * 8);
    double ss[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        ss[q] = 0.0;
#pragma unroll
        for (int i = 0; i < 8; ++i) ss[q] += (double)v[q][i] * (double)v[q][i];
    }
    double t = (ss[0] + ss[2]) + (ss[1] + ss[3]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t += __shfl_down(t, o);
    const float mean_sq = (float)(lane_f64(t, 0) / 2048.0);
    const float r = 1.0f / sqrtf(mean_sq + f.eps);
    if (l == 0) inv[w] = r;
    __syncthreads();
    const float s = inv[n & 7];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t a = (uint32_t)wt[j][e >> 1], b = (uint32_t)wt[j][2 + (e >> 1)];
            xa[j][e] = (xa[j][e] * s) * __uint_as_float(e & 1 ? a & 0xffff0000u : a << 16);
            xb[j][e] = (xb[j][e] * s) * __uint_as_float(e & 1 ? b & 0xffff0000u : b << 16);
        }
    __syncthreads();  // inv lies in the products' reduction buffer
}

// The q_proj | kv_a projection block of k_gemv_ksplit<1, 1> with this workgroup's index (B <= 8
// sequences, in = 2048, the same XCD-aware block -> (row block, k quarter) map), by the 512
// threads of a fused attention workgroup: wave w does that kernel's waves w and w + 8 (k-blocks
// kq 512 + 32 w and + 256), and the sixteen products are summed through LDS in that kernel's
// wave order, in two halves (lds: 32 KB), so the partials written to y equal its outputs bit for
// bit. They are stored with device-scope stores (read on other XCDs in this launch), and the
// block counted on its head's counter (q rows: 192 per head) or the kv_a counter (index 16).
// Called by both roles before any history request: its loads are then first in the CU's queue
// and its waits cover nothing else. (Measured on the headline step: with the task on the score
// waves only and the mix waves' history requests issued beside it, 1.404 ms against 1.378 ms.)
template <bool NORM>
__device__ __forceinline__ void fq_gemv(const FqArgs &f, int B, uint8_t *lds) {
    const int i = blockIdx.x;
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
    const int xcd = i & 7, rb = 2 * (i >> 3) + (xcd & 1);
    const int out = f.out0 + f.out1, kq = xcd >> 1, row0 = rb * 64, part = n >> 3;
    if (!f.gemv || i >= kGemvTasks || row0 >= out) return;  // uniform per workgroup
    v4f(*red)[4][64] = (v4f(*)[4][64])lds;                  // [8][4][64]
    const uint16_t *wr[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int row = min(row0 + 16 * t + n, out - 1);  // rows past the end are never stored
        wr[t] = row < f.out0 ? f.wq + (size_t)row * f.in : f.wkva + (size_t)(row - f.out0) * f.in;
    }
    v4i wa[2][4];
    v4f xa[2], xb[2];
    const float *xr = f.x + (size_t)min(n & 7, B - 1) * f.ldx;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int kbase = kq * 512 + (w + 8 * j) * 32 + g * 8;
#pragma unroll
        for (int t = 0; t < 4; ++t) wa[j][t] = __builtin_nontemporal_load((const v4i *)(wr[t] + kbase));
        xa[j] = *(const v4f *)(xr + kbase);
        xb[j] = *(const v4f *)(xr + kbase + 4);
    }
    if (NORM) fq_norm_x(f, B, kq, xa, xb, (float *)lds);
    v4f acc[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const v8bf xv = split8_part(xa[j], xb[j], part);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            acc[j][t] = mfma_bf16(__builtin_bit_cast(v8bf, wa[j][t]), xv, v4f{0.f, 0.f, 0.f, 0.f});
    }
    v4f s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int t = 0; t < 4; ++t) red[w][t][l] = acc[j][t];
        __syncthreads();
        if (w < 4) {
            // wave t sums row tile t over the sixteen waves in order (waves 8 j .. 8 j + 7 here)
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                if (j == 0 && q == 0) s = red[0][w][l];
                else s += red[q][w][l];
            }
        }
        __syncthreads();
    }
    if (w < 4) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += dpp_f32<0x128>(s[e]);  // row_ror:8 = lane ^ 8
        if (n < 8 && n < B) {
            float *y = f.y + (size_t)kq * f.pstride + (size_t)n * f.ldy;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = row0 + 16 * w + 4 * g + e;
                if (r < out) st_sc1_b32(y + r, __float_as_uint(s[e]));
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stores have reached memory
    }
    __syncthreads();
    if (tid == 0)
        __hip_atomic_fetch_add(fq_gflag(f, row0 < f.out0 ? row0 / 192 : 16), 1u, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
}

// Query of (sequence b, head h): qprep_body's Q8 path for R = 512, DN = 128, DR = 64, QD = 192
// over 8 waves (wave w: latent tiles 4 (w & 1) .. +3 of qprep_body's wave w >> 1). scr: 2848 B.
__device__ __forceinline__ void fq_qprep(const FqArgs &f, const AttnHot &hh, const SeqDesc &s, int b, int h,
                                         uint8_t *scr) {
    float *qn = (float *)scr, *qr = qn + 128, *ql = qr + 64, *red = ql + 512;
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
    const int w4 = w >> 1, t0 = 4 * (w & 1);
    const uint16_t *ut = f.ukt + ((size_t)(h * 4 + w4) * 32 * 64 + l) * 8;
    v8bf wa[4][4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) wa[tt][ks] = *(const v8bf *)(ut + (size_t)((t0 + tt) * 4 + ks) * 64 * 8);
    const float *qh = f.y + (size_t)b * f.ldy + (size_t)h * 192;
    if (f.gemv) fq_wait_all(f, fq_gflag(f, h), 12u);  // the 3 row blocks x 4 k quarters of head h
    if (tid < 192) {
        const float v = sum_parts(qh + tid, kGemvKs, f.pstride);
        if (tid < 128) qn[tid] = v;
        else qr[tid - 128] = v;
    }
    const float2 csv = tid < 32 ? f.cs[(size_t)s.pos * 32 + tid] : float2{0.f, 0.f};
    __syncthreads();
    const int m0 = n == 0 ? -1 : 0, m1 = n == 1 ? -1 : 0;
    v8bf qb[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const v4f x0 = *(const v4f *)(qn + 32 * ks + 8 * g), x1 = *(const v4f *)(qn + 32 * ks + 8 * g + 4);
        v8bf hi, lo;
        split8_cvt(x0, x1, hi, lo);
        const v4i hv = __builtin_bit_cast(v4i, hi), lv = __builtin_bit_cast(v4i, lo);
        qb[ks] = __builtin_bit_cast(v8bf, (hv & m0) | (lv & m1));
    }
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
        v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) acc = mfma_bf16(wa[tt][ks], qb[ks], acc);
        v4f v;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = acc[i] + dpp_f32<0xB1>(acc[i]);  // quad_perm [1,0,3,2]
        if (n == 0) {
            const int r = 128 * w4 + 16 * (t0 + tt) + 4 * g;
#pragma unroll
            for (int i = 0; i < 4; ++i) ql[r + i] = v[i];
        }
    }
    if (tid < 32) {
        const int i = tid;
        const float ev = qr[2 * i], od = qr[2 * i + 1];
        const float ec = ev * csv.x, os = od * csv.y, oc = od * csv.x, es = ev * csv.y;
        const float r0 = ec - os, r1 = oc + es;
        const size_t o = ((size_t)b * 16 + h) * 64;
        const float qsc = 1.0f / sqrtf(192.0f);
        uint16_t hi, lo;
        split_bf16(r0 * qsc, hi, lo);
        st_sc1_b16((void *)(hh.qrhi + o + i), hi);
        st_sc1_b16((void *)(hh.qrlo + o + i), lo);
        split_bf16(r1 * qsc, hi, lo);
        st_sc1_b16((void *)(hh.qrhi + o + 32 + i), hi);
        st_sc1_b16((void *)(hh.qrlo + o + 32 + i), lo);
    }
    __syncthreads();
    float m = 0.f;
    v4f qv = {0.f, 0.f, 0.f, 0.f};
    if (tid < 128) {
        qv = *(const v4f *)(ql + 4 * tid);
#pragma unroll
        for (int i = 0; i < 4; ++i) m = fmaxf(m, fabsf(qv[i]));
    }
    const float amax = block512_max(m, red);
    const bool ok = amax > 0.f && isfinite(amax);
    const float inv = ok ? 127.0f / amax : 0.f;
    if (tid < 128) {
        uint32_t ph = 0, pl = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float v = qv[i] * inv;
            float hi = rintf(v);
            hi = fminf(fmaxf(hi, -127.f), 127.f);
            float lo = rintf((v - hi) * 254.0f);
            lo = fminf(fmaxf(lo, -127.f), 127.f);
            ph |= (uint32_t)(uint8_t)(int8_t)hi << (8 * i);
            pl |= (uint32_t)(uint8_t)(int8_t)lo << (8 * i);
        }
        const size_t o = ((size_t)b * 16 + h) * 512 + 4 * tid;
        st_sc1_b32((void *)(hh.qhi + o), ph);
        st_sc1_b32((void *)(hh.qlo + o), pl);
    }
    if (tid == 0) st_sc1_b32((void *)(hh.qs + (size_t)b * 16 + h), __float_as_uint(ok ? amax / 127.0f : 0.f));
}

// Row of sequence b: append_body's Q8 path for R = 512, DR = 64 over 8 waves (the RMSNorm sum
// over the first 256 threads, two values each, as there). scr: 4448 B.
__device__ __forceinline__ void fq_append(const FqArgs &f, const SeqDesc &s, int b, uint8_t *scr) {
    float *kat = (float *)scr, *lat = kat + 576;
    double *redd = (double *)(lat + 512);
    float *redf = (float *)(redd + 8);
    const int tid = threadIdx.x, pos = s.pos;
    const float *ky = f.y + (size_t)b * f.ldy + f.koff;
    if (f.gemv) fq_wait_all(f, fq_gflag(f, 16), 36u);  // the 9 kv_a row blocks x 4 k quarters
    const float kv0 = sum_parts(ky + tid, kGemvKs, f.pstride);
    const float kv1 = tid < 64 ? sum_parts(ky + 512 + tid, kGemvKs, f.pstride) : 0.f;
    const float nw = bf16_to_f32(f.norm[tid]);
    const float2 csv = tid < 32 ? f.cs[(size_t)pos * 32 + tid] : float2{0.f, 0.f};
    kat[tid] = kv0;
    if (tid < 64) kat[512 + tid] = kv1;
    __syncthreads();
    double ss = 0.0;
    if (tid < 256) {
        for (int r = tid; r < 512; r += 256) {
            const double v = (double)kat[r];
            ss += v * v;
        }
    }
    const float mean_sq = (float)(block512_sum_f64(ss, redd) / 512.0);
    const float inv = 1.0f / sqrtf(mean_sq + f.eps);
    const float t = kat[tid] * inv;
    lat[tid] = t * nw;
    __syncthreads();
    const float amax = block512_max(fmaxf(0.f, fabsf(lat[tid])), redf);
    const bool zero = !(amax > 0.0f) || !isfinite(amax);
    const float scale = zero ? 1.0f : amax / 127.0f;
    const float qinv = zero ? 0.0f : 1.0f / scale;
    uint8_t *row_out = f.rows + (size_t)b * f.row_bytes;
    if (tid < 128) {
        uint32_t pk = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int8_t q = 0;
            if (!zero) {
                float v = roundf(lat[4 * tid + i] * qinv);
                v = v > 127.0f ? 127.0f : v;
                v = v < -127.0f ? -127.0f : v;
                q = (int8_t)v;
            }
            pk |= (uint32_t)(uint8_t)q << (8 * i);
        }
        st_sc1_b32((int8_t *)s.a + (size_t)pos * 512 + 4 * tid, pk);
        *(uint32_t *)(row_out + 4 * tid) = pk;
    }
    if (tid == 0) {
        st_sc1_b32((float *)s.b + pos, __float_as_uint(scale));
        *(float *)(row_out + 512) = scale;
    }
    if (tid < 32) {
        const int i = tid;
        const float ev = kat[512 + 2 * i], od = kat[512 + 2 * i + 1];
        const float ec = ev * csv.x, os = od * csv.y, oc = od * csv.x, es = ev * csv.y;
        const uint16_t h0 = f32_to_bf16_rne(ec - os), h1 = f32_to_bf16_rne(oc + es);
        uint16_t *rp = (uint16_t *)s.c + (size_t)pos * 64;
        st_sc1_b16(rp + i, h0);
        st_sc1_b16(rp + 32 + i, h1);
        uint16_t *ro = (uint16_t *)(row_out + 516);
        ro[i] = h0;
        ro[32 + i] = h1;
    }
}

// The producer task of this workgroup, if any (blocks [0, 17 B)), then its flag. Called by both
// roles of the Q8 kernel at the same point of their barrier sequences (uniform per workgroup).
__device__ __forceinline__ void fq_produce(const AttnArgs &a, const AttnHot &hh, uint8_t *scr) {
    const int i = blockIdx.x, B = hh.nseq;
    if (i >= 17 * B) return;
    const DescLane dl = desc_lane(a.t);
    const int b = i < 16 * B ? i >> 4 : i - 16 * B;
    const SeqDesc s = desc_pick(dl, b);
    if (i < 16 * B) fq_qprep(a.fq, hh, s, b, i & 15, scr);
    else fq_append(a.fq, s, b, scr);
    if (threadIdx.x < 128) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the storing waves
    __syncthreads();
    if (threadIdx.x == 0)
        __hip_atomic_fetch_add(i < 16 * B ? fq_qflag(a.fq, b) : fq_aflag(a.fq, b), 1u, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
}

// Position of the quantised weight of (head h, chunk row r) within one level: 16-byte groups
// of rows XOR-swizzled by the head, so the mix waves' 16-byte reads (one head, 16 rows per lane)
// spread over the banks.
__device__ __forceinline__ int q8_wpos(int h, int r) { return h * kQ8Ws + ((((r >> 4) ^ (h >> 1)) & 3) << 4) + (r & 15); }

// Slot swizzle of the code rows: physical 16-byte slot = logical slot ^ q8_swz(row).
__device__ __forceinline__ int q8_swz(int row) { return (row & 7) ^ (((row >> 4) & 1) << 2); }

// Maxima over the 16 lanes of each DPP row for four values: one v_max_f32_dpp per step and
// value (quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_ror:4, row_ror:8), the four chains
// interleaved so that each DPP source was written at least three instructions earlier.
__device__ __forceinline__ void row16_max4(float &a, float &b, float &c, float &d) {
    asm volatile(
        "s_nop 1\n\t"
        "v_max_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %3, %3, %3 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %3, %3, %3 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %2, %2, %2 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %3, %3, %3 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %1, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %2, %2, %2 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32_dpp %3, %3, %3 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1"
        : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}

// ds_read_b64_tr_b8: within each 16-lane group, destination lane j byte i comes from the
// 8 bytes addressed by source lane 2i + (j >> 3), at byte j & 7.
__device__ __forceinline__ v2i lds_read_tr8(const uint8_t *p) {
    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i *)(p));
}

// The three-level quantised weights of this lane's row (rowl) for heads 4g .. 4g+3:
// v = p * s * wscale in [0, 127] ~= hi + lo/254 + lo2/254^2.
__device__ __forceinline__ void put_q8_weights(int8_t *wqc, const float *pv, float swj, int g, int rowl) {
    int qhv[4], qlv[4], q2v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float v = pv[i] * swj;
        const float hi = fminf(rintf(v), 127.f);
        // v - hi is exact (|v - hi| <= 1/2): lo and lo2 span the int8 range
        const float r1 = (v - hi) * 254.0f;
        const float lo = rintf(r1);
        qhv[i] = (int)hi;
        qlv[i] = (int)lo;
        q2v[i] = (int)rintf((r1 - lo) * 254.0f);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int o = q8_wpos(4 * g + i, rowl);
        wqc[o] = (int8_t)qhv[i];
        wqc[16 * kQ8Ws + o] = (int8_t)qlv[i];
        wqc[32 * kQ8Ws + o] = (int8_t)q2v[i];
    }
}


// The two roles run separate code (their registers do not overlap) with the same sequence of
// workgroup barriers: two in the prologue (P0: the query operands, copied once by DMA into code
// slot 3, have landed, and only chunk 0 is requested ahead of them; P: chunk 0 has landed, and the
// score waves have read the query out of slot 3, which the chunk-3 DMA of step 0 then
// overwrites), per step k = 0 .. nch one (A) plus two more (B, C) when the flags read after A ask
// for an exchange, and one at the end. Every wave reads the
// same LDS flags after A, so all eight take the same barriers. Everything the score waves read
// per chunk (codes, RoPE keys, scales) arrives in LDS by the mix waves' DMA, so their steps
// never wait on global-memory latency.
// Combine modes of the Q8 launch (FqArgs::comb): none; XCD-local (every split of a sequence on
// one XCD, partials read from its L2); across XCDs (partials stored with device-scope stores,
// read from memory).
enum { kCombNone = 0, kCombXcd = 1, kCombCross = 2 };
template <bool FUSE, int COMB, bool NORM>  // FUSE: the launch also prepares the queries and appends the rows (fq_produce)
__device__ __forceinline__ void q8_score_role(const AttnArgs &a, const AttnHot &h, const SeqDesc &sd, uint8_t *smem, int w, int b,
                                              int r0, int r1, int nch, int sid, int cpos) {
    int8_t *wq = (int8_t *)(smem + kQ8WqOff);
    int *oflag = (int *)(smem + kQ8FlagOff);
    float *mloc = (float *)(smem + kQ8MlOff);
    float *abuf = (float *)(smem + kQ8AlOff);
    float *lsum = (float *)(smem + kQ8LsOff);
    float *smx = (float *)(smem + kQ8SmOff);
    const int tid = threadIdx.x, l = tid & 63, n = l & 15, g = l >> 4;
    const float *gscl = (const float *)sd.b;
    const int rowl = 16 * w + n;  // chunk row of this lane
    int sc_base[2], rp_off[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        sc_base[kb] = rowl * 512 + 16 * ((4 * kb + g) ^ q8_swz(rowl));
        rp_off[kb] = rowl * 128 + 16 * ((4 * kb + g) ^ (rowl & 7));
    }
    // query operands (A of the score MFMAs: head n, k slice 16g .. 16g+15 of each 64-wide block)
    // and the split's largest row scale: all loads issued before the first wait
    v4i qh[8], ql[8];
    v8bf qrh[2], qrl[2];
    float qsd[4], m_run[4], l_lane[4];
    if constexpr (FUSE) {
        // this workgroup's projection task (FqArgs::gemv; LDS: code slot 3, free until the
        // query copy after Q), its producer task, then (one poller, barrier Q) the 16 query heads
        // of its sequence and, where the split holds the new row (whose scale the loads below
        // read and whose chunk the mix waves request after Q), that row
        fq_gemv<NORM>(a.fq, h.nseq, smem + 3 * kQ8CodeB);
        fq_produce(a, h, smem + kQ8WqOff);
        if (w == 0) {
            fq_wait(a.fq, fq_qflag(a.fq, b), 16u);
            if (cpos >= 0) fq_wait(a.fq, fq_aflag(a.fq, b), 1u);
        }
        lds_barrier();  // Q
    }
    // the query's int8 scales first: the first chunk's scores need them right after P (written in
    // this launch when FUSE: read past the L2, whose line may hold another sequence's scales)
    float qsr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) qsr[i] = FUSE ? ld_sc1_f32(h.qs + (size_t)b * 16 + 4 * g + i) : h.qs[(size_t)b * 16 + 4 * g + i];
    // the sequence's query operands (hi, lo codes: 8 KB each; RoPE hi, lo: 2 KB each) once into
    // code slot 3 by DMA (wave w: 1 KB pieces 5w .. 5w+4), read from there by all four waves
    const uint32_t qslot = lds_addr(smem) + 3 * kQ8CodeB;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const int p = 5 * w + i;
        const int8_t *src = p < 8 ? h.qhi + (size_t)b * 8192 + p * 1024
                          : p < 16 ? h.qlo + (size_t)b * 8192 + (p - 8) * 1024
                          : p < 18 ? (const int8_t *)(h.qrhi + (size_t)b * 1024) + (p - 16) * 1024
                                   : (const int8_t *)(h.qrlo + (size_t)b * 1024) + (p - 18) * 1024;
        dma_b128(src + 16 * l, qslot + (uint32_t)(p * 1024));
    }
    {
        const int nr = r1 - r0;
        float sv[8];
        // rows past the split end re-read its last row (a duplicate does not change the max)
#pragma unroll
        for (int i = 0; i < 8; ++i) sv[i] = gscl[r0 + min(tid + 256 * i, nr - 1)];
        wait_vm(8);     // this wave's query pieces have landed (the 8 scale loads may not have)
        lds_barrier();  // P0
        {
            const uint8_t *qb = smem + 3 * kQ8CodeB;
#pragma unroll
            for (int kb = 0; kb < 8; ++kb) {
                qh[kb] = *(const v4i *)(qb + n * 512 + 64 * kb + 16 * g);
                ql[kb] = *(const v4i *)(qb + 8192 + n * 512 + 64 * kb + 16 * g);
            }
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                qrh[kb] = *(const v8bf *)(qb + 16384 + 2 * (n * 64 + 8 * (4 * kb + g)));
                qrl[kb] = *(const v8bf *)(qb + 18432 + 2 * (n * 64 + 8 * (4 * kb + g)));
            }
        }
        // the loads complete after P0: the mix waves' first DMA is not held up by them (without
        // this the compiler may compute the max, and so wait for the loads, before the barrier)
#pragma unroll
        for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(sv[i]));
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) m = fmaxf(m, sv[i]);
        for (int r = tid + 2048; r < nr; r += 256) m = fmaxf(m, gscl[r0 + r]);
        m = wave_max(m);
        if (l == 0) smx[w] = m;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        qsd[i] = qsr[i] * (a.smscale / 254.0f);
        m_run[i] = -INFINITY;
        l_lane[i] = 0.f;
    }
    lds_barrier();  // P: chunk 0 has landed; the split's largest scale is published
    // largest row scale of the split: the common bound of the quantised weights
    const float smax = fmaxf(fmaxf(smx[0], smx[1]), fmaxf(smx[2], smx[3]));
    const float wscale = smax > 0.f ? 127.0f / (kQ8Pmax * smax) : 0.f;

    for (int k = 0; k <= nch; ++k) {
        const int par = k & 1;
        int *fl_out = oflag + 4 * par;
        float *ml = mloc + 64 * par;
        int8_t *wqc = wq + par * kQ8WqB;  // weights of chunk k
        float sc[4], pv[4], sj = 0.f;
        if (k < nch) {
            const uint8_t *buf = smem + (k % kQ8Ring) * kQ8CodeB;
            const uint8_t *rbuf = smem + kQ8RopeOff + (k % kQ8RRing) * kQ8RSlot;
            const int base = r0 + k * kQ8Ch;
            v4i bv[8];
            v8bf rv[2];
#pragma unroll
            for (int kb = 0; kb < 8; ++kb) bv[kb] = *(const v4i *)(buf + sc_base[kb & 1] + 128 * (kb >> 1));
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) rv[kb] = *(const v8bf *)(rbuf + rp_off[kb]);
            sj = ((const float *)(rbuf + kQ8RopeB))[rowl];
            v4i ih = {0, 0, 0, 0}, il = {0, 0, 0, 0};
            v4f fr = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < 8; ++kb) {
                ih = mfma_i8(qh[kb], bv[kb], ih);
                il = mfma_i8(ql[kb], bv[kb], il);
            }
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                fr = mfma_bf16(qrh[kb], rv[kb], fr);
                fr = mfma_bf16(qrl[kb], rv[kb], fr);
            }
            const bool valid = base + rowl < r1;
            bool over = false;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // 254 ih + il is exact in int32 (|ih|, |il| <= 512 * 127 * 127, so |254 ih + il|
                // <= 2.106e9 < 2^31); qsd carries the 1/254
                const float dot = (float)(ih[i] * 254 + il[i]);
                const float sv = fmaf(qsd[i] * sj, dot, fr[i]);
                sc[i] = valid ? sv : -INFINITY;
                // weights against the current reference max; a row above it by more than
                // ln kQ8Pmax (every valid row of the first chunk, where it is -inf) sends the
                // block through the exchange below
                over |= sc[i] > m_run[i] + kQ8LnPmax;
                pv[i] = __expf(sc[i] - m_run[i]);
            }
            put_q8_weights(wqc, pv, sj * wscale, g, rowl);
            const bool wover = __any(over);
            if (l == 0) fl_out[w] = wover ? 1 : 0;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[i] = pv[i] = 0.f;
            if (l == 0) fl_out[w] = 0;  // the mix waves' last step: nothing to exchange
        }
        lds_barrier();  // A
        const v4i fl = *(const v4i *)fl_out;
        if ((fl.x | fl.y | fl.z | fl.w) != 0) {
            // Some row of chunk k exceeds the reference max: exchange the chunk maxima, move the
            // reference max of the heads concerned, quantise the chunk's weights again and
            // publish alpha for the mix waves (they rescale before adding chunk k). The first
            // finite maximum of a head needs no rescale (nothing is accumulated before it).
            float lm[4] = {sc[0], sc[1], sc[2], sc[3]};
            row16_max4(lm[0], lm[1], lm[2], lm[3]);
            if (n == 0) *(v4f *)(ml + w * 16 + 4 * g) = v4f{lm[0], lm[1], lm[2], lm[3]};
            lds_barrier();  // B
            const v4f mw0 = *(const v4f *)(ml + 4 * g), mw1 = *(const v4f *)(ml + 16 + 4 * g);
            const v4f mw2 = *(const v4f *)(ml + 32 + 4 * g), mw3 = *(const v4f *)(ml + 48 + 4 * g);
            float alpha[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float cm = fmaxf(fmaxf(mw0[i], mw1[i]), fmaxf(mw2[i], mw3[i]));
                const bool mv = cm > m_run[i] + kQ8LnPmax;
                const bool rs = mv && m_run[i] != -INFINITY;
                const float mnew = mv ? cm : m_run[i];
                alpha[i] = rs ? __expf(m_run[i] - mnew) : 1.0f;
                m_run[i] = mnew;
                pv[i] = __expf(sc[i] - mnew);
                l_lane[i] *= alpha[i];
            }
            put_q8_weights(wqc, pv, sj * wscale, g, rowl);
            if (w == 0 && n == 0) *(v4f *)(abuf + 16 * par + 4 * g) = v4f{alpha[0], alpha[1], alpha[2], alpha[3]};
            lds_barrier();  // C
        }
        if (k < nch)
#pragma unroll
            for (int i = 0; i < 4; ++i) l_lane[i] += pv[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) l_lane[i] = row16_sum(l_lane[i]);
    if (n == 0)
#pragma unroll
        for (int i = 0; i < 4; ++i) lsum[w * 16 + 4 * g + i] = l_lane[i];
    lds_barrier();  // end
    if (w == 0 && n == 0) {
        float *P = h.part + (size_t)sid * 16 * 514;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int hh = 4 * g + i;
            const float lv = (lsum[hh] + lsum[16 + hh]) + (lsum[32 + hh] + lsum[48 + hh]);
            if constexpr (COMB == kCombCross) {  // read on other XCDs in this launch
                st_sc1_b32(&P[8192 + hh], __float_as_uint(m_run[i]));
                st_sc1_b32(&P[8192 + 16 + hh], __float_as_uint(lv));
            } else {
                P[8192 + hh] = m_run[i];
                P[8192 + 16 + hh] = lv;
            }
        }
    }
}

template <bool ONCE, bool FUSE, int COMB, bool NORM>
__device__ __forceinline__ void q8_mix_role(const AttnArgs &a, const AttnHot &h, const SeqDesc &sd, uint8_t *smem, int mw, int b,
                                            int r0, int r1, int nch, int sid, int cpos) {
    const int8_t *wq = (const int8_t *)(smem + kQ8WqOff);
    const int *oflag = (const int *)(smem + kQ8FlagOff);
    const float *abuf = (const float *)(smem + kQ8AlOff);
    const float *smx = (const float *)(smem + kQ8SmOff);
    const uint32_t sbase = lds_addr(smem);
    const int l = threadIdx.x & 63, n = l & 15, g = l >> 4;
    const int8_t *gcodes = (const int8_t *)sd.a;
    const float *gscl = (const float *)sd.b;
    const uint16_t *grope = (const uint16_t *)sd.c;
    constexpr bool once = ONCE;
    // DMA plan. Codes: mix wave mw copies row pairs 8mw .. 8mw+7 of a chunk; lane l of
    // instruction k takes row 2(8mw + k) + (l >> 5), physical slot l & 31 (logical slot
    // (l & 31) ^ swz). RoPE keys: instruction k of wave mw covers rows 8(2mw + k) .. +7, lane l
    // row 8(2mw + k) + (l >> 3), physical slot l & 7 (logical (l & 7) ^ (row & 7)). Scales: wave
    // 0, lane l row l. Rows past the split end (last chunk only) re-read the split's last row
    // (in bounds); their weights are 0.
    int code_off[8], rope_row[2], rope_el[2];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int row = 2 * (mw * 8 + k) + (l >> 5);
        code_off[k] = row * 512 + 16 * ((l & 31) ^ q8_swz(row));
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int row = 8 * (2 * mw + k) + (l >> 3);
        rope_row[k] = row;
        rope_el[k] = 8 * ((l & 7) ^ (row & 7));
    }
    const int nrope = mw == 0 ? 3 : 2;  // DMA instructions per chunk for keys + scales
    auto issue_codes = [&](int c) __attribute__((always_inline)) {
        const uint32_t buf = sbase + (uint32_t)((c % kQ8Ring) * kQ8CodeB);
        const int rb0 = r0 + c * kQ8Ch;
        if (rb0 + kQ8Ch <= r1) {
            const int8_t *gc = gcodes + (size_t)rb0 * 512;
#pragma unroll
            for (int k = 0; k < 8; ++k) dma_hist_b128(gc + code_off[k], buf + (uint32_t)((mw * 8 + k) * 1024), once);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int row = code_off[k] >> 9;
                const int gro = min(rb0 + row, r1 - 1);
                dma_hist_b128(gcodes + (size_t)gro * 512 + (code_off[k] & 511), buf + (uint32_t)((mw * 8 + k) * 1024), once);
            }
        }
    };
    auto issue_rope = [&](int c) __attribute__((always_inline)) {
        const uint32_t buf = sbase + (uint32_t)(kQ8RopeOff + (c % kQ8RRing) * kQ8RSlot);
        const int rb0 = r0 + c * kQ8Ch;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int gro = min(rb0 + rope_row[k], r1 - 1);
            dma_hist_b128(grope + (size_t)gro * 64 + rope_el[k], buf + (uint32_t)((2 * mw + k) * 1024), once);
        }
        if (mw == 0) dma_hist_b32(gscl + min(rb0 + l, r1 - 1), buf + (uint32_t)kQ8RopeB, once);
    };
    // transposed reads: rows 16g + (n >> 1) and 16g + 8 + (n >> 1) share the swizzle (+4096)
    int tr_off[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const int row = 16 * g + (n >> 1);
        tr_off[t] = row * 512 + 16 * ((8 * mw + t) ^ q8_swz(row)) + 8 * (n & 1);
    }
    const int wq_off = n * kQ8Ws + (((g ^ (n >> 1)) & 3) << 4);  // q8_wpos(n, 16 g)
    v4i ahi[8], alo[8], alo2[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        ahi[t] = v4i{0, 0, 0, 0};
        alo[t] = v4i{0, 0, 0, 0};
        alo2[t] = v4i{0, 0, 0, 0};
    }
    // prologue: codes of chunks 0 .. 2 and keys of chunks 0, 1 in flight, chunk 0 first (beside
    // the score waves' query DMA, before P0) and the rest after it; the issue order codes(c+1)
    // before keys(c) keeps the per-step wait count below uniform
    if constexpr (!FUSE) {
        issue_codes(0);
        issue_rope(0);
        lds_barrier();  // P0
        if (nch > 1) issue_codes(1);
        if (nch > 2) issue_codes(2);
        if (nch > 1) issue_rope(1);
    } else {
        // The same requests in the same order (codes 0, keys 0, codes 1, codes 2, keys 1), as many
        // as possible ahead of barrier Q (the queries and the new row are ready, polled by score
        // wave 0): a producer issues them after its task (its own loads go first), the others
        // before it; from the first that touches the chunk holding the new row (cpos) on they
        // wait for Q. Measured against chunk 0 only ahead of Q (headline step 1.510 ms): all
        // three chunks before the task 1.490 ms, a producer's after its task 1.483 ms.
        auto issue_item = [&](int it) __attribute__((always_inline)) {
            if (it == 0) issue_codes(0);
            else if (it == 1) issue_rope(0);
            else if (it == 2) { if (nch > 1) issue_codes(1); }
            else if (it == 3) { if (nch > 2) issue_codes(2); }
            else if (nch > 1) issue_rope(1);
        };
        int it = 0;
        auto issue_ahead = [&]() __attribute__((always_inline)) {
            for (; it < 5; ++it) {
                const int ch = it < 2 ? 0 : it == 2 ? 1 : it == 3 ? 2 : 1;
                if (cpos >= 0 && ch >= cpos) break;
                issue_item(it);
            }
        };
        const bool prod = (int)blockIdx.x < 17 * h.nseq;
        // a projection task goes before the history requests (fq_gemv)
        fq_gemv<NORM>(a.fq, h.nseq, smem + 3 * kQ8CodeB);
        if (!prod) issue_ahead();
        fq_produce(a, h, smem + kQ8WqOff);
        if (prod) issue_ahead();
        lds_barrier();  // Q
        for (; it < 5; ++it) issue_item(it);
        lds_barrier();  // P0
    }
    wait_vm(nch > 1 ? (nch > 2 ? 16 : 8) + nrope : 0);
    lds_barrier();  // P
    const float smax = fmaxf(fmaxf(smx[0], smx[1]), fmaxf(smx[2], smx[3]));
    bool pend = false;  // a reference max moved in the previous step: rescale before mixing
    v4i bt[8];          // chunk k-1's codes, transposed (read in step k-1)
    for (int k = 0; k <= nch; ++k) {
        const int par = k & 1;
        // codes of chunk k+3 into the slot of chunk k-1 and keys of chunk k+2 into the slot of
        // chunk k-1: every wave finished reading both before the previous barrier
        if (k + 3 < nch) issue_codes(k + 3);
        if (k + 2 < nch) issue_rope(k + 2);
        if (k >= 1) {
            if (pend) {
                // (254^2 hi + 254 lo + lo2) * alpha, level by level in double (the products are
                // exact), each level's rounding remainder carried into the next
                const v4f al4 = *(const v4f *)(abuf + 16 * (par ^ 1) + 4 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (al4[i] == 1.0f) continue;
                    const double al = (double)al4[i];
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        const double h = (double)ahi[t][i] * al, hr = rint(h);
                        const double o = (h - hr) * 254.0 + (double)alo[t][i] * al, orr = rint(o);
                        const double o2 = (o - orr) * 254.0 + (double)alo2[t][i] * al;
                        ahi[t][i] = (int)hr;
                        alo[t][i] = (int)orr;
                        alo2[t][i] = (int)rint(o2);
                    }
                }
            }
            // chunk k-1 with its weights (written by the score waves in step k-1)
            const int8_t *wqp = wq + (par ^ 1) * kQ8WqB;
            const v4i wh = *(const v4i *)(wqp + wq_off);
            const v4i wl = *(const v4i *)(wqp + 16 * kQ8Ws + wq_off);
            const v4i wl2 = *(const v4i *)(wqp + 32 * kQ8Ws + wq_off);
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                ahi[t] = mfma_i8(wh, bt[t], ahi[t]);
                alo[t] = mfma_i8(wl, bt[t], alo[t]);
                alo2[t] = mfma_i8(wl2, bt[t], alo2[t]);
            }
        }
        if (k < nch) {
            // chunk k (being scored in this step): codes transposed for the next step's mix
            const uint8_t *buf = smem + (k % kQ8Ring) * kQ8CodeB;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const v2i b0 = lds_read_tr8(buf + tr_off[t]);
                const v2i b1 = lds_read_tr8(buf + tr_off[t] + 4096);
                bt[t] = v4i{b0.x, b0.y, b1.x, b1.y};
            }
        }
        // codes and keys of chunk k+1 (scored in the next step) have landed before the barrier:
        // issued after the keys of chunk k+1 are only the codes of k+3 and the keys of k+2
        if (k + 1 < nch) wait_vm((k + 3 < nch ? 8 : 0) + (k + 2 < nch ? nrope : 0));
        lds_barrier();  // A
        const v4i fl = *(const v4i *)(oflag + 4 * par);
        pend = (fl.x | fl.y | fl.z | fl.w) != 0;
        if (pend) {
            lds_barrier();  // B
            lds_barrier();  // C
        }
    }
    lds_barrier();  // end
    // The partials are read once, by the combine, mostly on other XCDs: non-temporal stores
    // leave no dirty lines in this XCD's L2 for the end-of-kernel write-back (headline step:
    // attention 33.5 -> 32.7 us per launch; the combine, which then reads every partial from
    // memory, +0.15 us). In the BF16 and FP32 kernels the same stores made no difference
    // beyond the noise of the ragged legs (±2 %), and they keep plain stores.
    float *P = h.part + (size_t)sid * 16 * 514;
    const float wfac = kQ8Pmax * smax * (1.0f / (127.0f * 254.0f * 254.0f));
    // the lane's row and group formed again from the thread index (opaque to the compiler):
    // held across the chunk loop they cost the one register beyond the 256 of a wave (a spill)
    int tx = threadIdx.x;
    asm volatile("" : "+v"(tx));
    const int ne = tx & 15, ge = (tx & 63) >> 4;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        const int r = 128 * mw + 16 * t + ne;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float v = wfac * fmaf((float)ahi[t][i], 64516.0f, fmaf((float)alo[t][i], 254.0f, (float)alo2[t][i]));
            // read in this launch (q8_comb_tail): by this XCD's workgroups from its L2, or by any
            // XCD's past the L2s
            if constexpr (COMB == kCombXcd) P[(4 * ge + i) * 512 + r] = v;
            else if constexpr (COMB == kCombCross) st_sc1_b32(&P[(4 * ge + i) * 512 + r], __float_as_uint(v));
            else __builtin_nontemporal_store(v, &P[(4 * ge + i) * 512 + r]);
        }
    }
}

// Position of latent column c of the merged mix in the combine's LDS row: 16-byte groups XOR-
// swizzled by c / 32, so the 16 lanes of a W_UV row read distinct banks.
__device__ __forceinline__ int mx_pos(int c) { return c ^ (((c >> 5) & 7) << 2); }
constexpr int kCombPre = 8;  // split-partial loads a combine thread issues before its first wait

// ---- the combine inside the Q8 attention launch ----------------------------------------------
// With every split of a sequence on one XCD (seq_of<true>), its split partials are in that XCD's
// L2 when the last split ends: each workgroup stores its partial with plain stores, waits until
// the L2 has acknowledged them (vmcnt) and counts itself on the sequence's counter; workgroup
// `split` < 32 then waits for the count to reach ns and combines (head split / 2, half split %
// 2) -- and further tasks split + ns, ... when ns < 32 -- with the arithmetic of k_combine_r512,
// whose launch this replaces. Its first read of a partial line comes after the wait (the CU has
// not read those lines in this launch, so its L1 holds no copy, and the launch began with the
// caches invalidated): the read is served by the L2. (Polling a line that the CU keeps reading
// does not work that way: the L1 keeps serving its first copy even with the sc0 bit on the load
// or a buffer_inv sc0 before it, measured with per-split done words in one line, whose wait
// never ended.) The counter (64 bits, one 128-byte line per sequence, after the query and row
// flags, cleared before each fused launch) is updated and polled with atomics, which are not
// served by the L1, and has one byte per XCC: a workgroup adds 1 << 8 * (its XCC id), so the waiters also see
// that all the sequence's splits ran on one XCC, which the placement assumes (workgroup i on XCD
// i % 8 + a per-launch offset); otherwise the partials would not all be in the reader's L2, and
// the launch raises FqArgs::err (results invalid) instead of reading them. The waits are bounded
// as fq_wait's are.
__device__ __forceinline__ unsigned long long *fq_cflag(const FqArgs &f, int b) {
    return (unsigned long long *)(f.flags + (size_t)kFqFlagStride * (2 * kMaxBatch + b));
}
__device__ __forceinline__ unsigned xcc_id() {
    unsigned x;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
    return x & 7;
}
// The counter's value by a returning atomic add of 0 (an atomic is never served from the L1).
__device__ __forceinline__ unsigned long long cnt_poll(unsigned long long *p) {
    unsigned long long v;
    asm volatile("global_atomic_add_x2 %0, %1, %2, off sc0\n\ts_waitcnt vmcnt(0)" : "=v"(v) : "v"(p), "v"(0ull) : "memory");
    return v;
}
// Sum of the eight byte fields (each <= ns <= 255, comb_ok).
__device__ __forceinline__ unsigned cnt_total(unsigned long long v) {
    unsigned t = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) t += (unsigned)(v >> (8 * i)) & 0xffu;
    return t;
}

// One (head h, half) of the combine of a sequence whose ns split partials start at P, by the
// 512 threads of the attention workgroup: thread t does the work of k_combine_r512's threads t
// and t + 512 in the same order (split groups sg and sg + 4; W_UV rows dd and dd + 32), so the
// outputs equal that kernel's bit for bit. wv: the thread's two W_UV row slices. lds: 27 KB.
__device__ __forceinline__ void comb_task(const float *P, float *ho, uint16_t *hos, int n, int HO, int b, int h,
                                          int half, int ns, const v4i (&wv)[2][4], uint8_t *lds) {
    constexpr int NH = 16;
    float *mx = (float *)lds;                      // 512 floats
    float *wts = mx + 512;                         // kMaxSplits floats
    v4f(*red)[128] = (v4f(*)[128])(wts + kMaxSplits);  // [8][128]
    float *sinv = (float *)(red + 8);
    const int tid = threadIdx.x;
    const int sg = __builtin_amdgcn_readfirstlane(tid >> 7);  // split groups sg and sg + 4
    const size_t stride = (size_t)NH * (512 + 2);
    int c4 = tid & 127;
    asm volatile("" : "+v"(c4));
    const float *Pm = P + (size_t)NH * 512 + h;
    float m0 = 0.f, l0 = 0.f;
    if (tid < 64) {
        const int i0 = min(tid, ns - 1);
        m0 = Pm[(size_t)i0 * stride];
        l0 = Pm[(size_t)i0 * stride + NH];
    }
    const float *Pg = P + (size_t)h * 512 + 4 * c4;
    v4f pre[2][kCombPre];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < kCombPre; ++i)
            pre[j][i] = sg + 4 * j + 8 * i < ns ? *(const v4f *)(Pg + (size_t)(sg + 4 * j + 8 * i) * stride)
                                                : v4f{0.f, 0.f, 0.f, 0.f};
    if (tid < 64) {
        float m = tid < ns ? m0 : -INFINITY;
        for (int i = tid + 64; i < ns; i += 64) m = fmaxf(m, Pm[(size_t)i * stride]);
        m = wave_max(m);
        float den = 0.f;
        if (tid < ns) {
            const float e = __expf(m0 - m);
            wts[tid] = e;
            den = l0 * e;
        }
        for (int i = tid + 64; i < ns; i += 64) {
            const float e = __expf(Pm[(size_t)i * stride] - m);
            wts[i] = e;
            den = fmaf(Pm[(size_t)i * stride + NH], e, den);
        }
        den = wave_sum(den);
        if (tid == 0) *sinv = 1.0f / den;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int g = sg + 4 * j;
        v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kCombPre; ++i) {
            const int sp = g + 8 * i;
            if (sp < ns) {
                const float wt = wts[sp];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = fmaf(pre[j][i][e], wt, acc[e]);
            }
        }
        for (int sp = g + 8 * kCombPre; sp < ns; sp += 8 * kCombPre) {
            v4f more[kCombPre];
#pragma unroll
            for (int i = 0; i < kCombPre; ++i)
                more[i] = sp + 8 * i < ns ? *(const v4f *)(Pg + (size_t)(sp + 8 * i) * stride) : v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < kCombPre; ++i) {
                if (sp + 8 * i < ns) {
                    const float wt = wts[sp + 8 * i];
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[e] = fmaf(more[i][e], wt, acc[e]);
                }
            }
        }
        red[g][c4] = acc;
    }
    __syncthreads();
    {
        const int cq = tid >> 2, e = tid & 3;
        float v = red[0][cq][e];
#pragma unroll
        for (int g8 = 1; g8 < 8; ++g8) v += red[g8][cq][e];
        mx[mx_pos(tid)] = v * *sinv;
    }
    __syncthreads();
    const int q = tid & 15;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int dd = 64 * half + 32 * r + (tid >> 4);
        float acc0 = 0.f, acc1 = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const v4f m0v = *(const v4f *)(mx + mx_pos(32 * q + 8 * c));
            const v4f m1v = *(const v4f *)(mx + mx_pos(32 * q + 8 * c + 4));
            const uint32_t u0 = (uint32_t)wv[r][c][0], u1 = (uint32_t)wv[r][c][1];
            const uint32_t u2 = (uint32_t)wv[r][c][2], u3 = (uint32_t)wv[r][c][3];
            acc0 = fmaf(__uint_as_float(u0 << 16), m0v.x, acc0);
            acc1 = fmaf(__uint_as_float(u0 & 0xffff0000u), m0v.y, acc1);
            acc0 = fmaf(__uint_as_float(u1 << 16), m0v.z, acc0);
            acc1 = fmaf(__uint_as_float(u1 & 0xffff0000u), m0v.w, acc1);
            acc0 = fmaf(__uint_as_float(u2 << 16), m1v.x, acc0);
            acc1 = fmaf(__uint_as_float(u2 & 0xffff0000u), m1v.y, acc1);
            acc0 = fmaf(__uint_as_float(u3 << 16), m1v.z, acc0);
            acc1 = fmaf(__uint_as_float(u3 & 0xffff0000u), m1v.w, acc1);
        }
        const float hsum = row16_sum(acc0 + acc1);  // the 16 lanes of row dd
        if (q == 0) {
            const size_t o = (size_t)b * HO + (size_t)h * 128 + dd;
            ho[o] = hsum;
            uint16_t hi, lo;
            split_bf16(hsum, hi, lo);
            hos[o] = hi;
            hos[(size_t)n * HO + o] = lo;
        }
    }
}

// The W_UV row slices of task (h, half) for comb_task (kv_b: [NH][DN + 128][512] bf16, DN = 128).
__device__ __forceinline__ void comb_wuv(const uint16_t *kv_b, int h, int half, v4i (&wv)[2][4]) {
    const int tid = threadIdx.x, q = tid & 15;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int dd = 64 * half + 32 * r + (tid >> 4);
        const uint16_t *row = kv_b + ((size_t)h * 256 + 128 + dd) * 512 + 32 * q;
#pragma unroll
        for (int c = 0; c < 4; ++c) wv[r][c] = *(const v4i *)(row + 8 * c);
    }
}

template <int COMB>
__device__ __forceinline__ void q8_comb_tail(const AttnArgs &a, const SeqDesc &s, int b, int split, uint8_t *smem) {
    constexpr int kTasks = 32;  // (head, half) pairs of 16 heads
    const int ns = s.nsplit, tid = threadIdx.x;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's partial stores are in the L2
    __syncthreads();
    unsigned long long *cf = fq_cflag(a.fq, b);
    const unsigned long long mine = 1ull << (8 * xcc_id());
    if (tid == 0) __hip_atomic_fetch_add(cf, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v4i wv[2][4];
    if (split < kTasks) comb_wuv(a.fq.kvb, split >> 1, split & 1, wv);  // requested before the wait
    if (tid == 0) {
        if (split < kTasks) {
            const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
            unsigned long long v;
            while (cnt_total(v = cnt_poll(cf)) < (unsigned)ns) {
                if (__builtin_amdgcn_s_memrealtime() - t0 > (uint64_t)a.fq.spin) break;
                __builtin_amdgcn_s_sleep(1);
            }
            // a timeout, or (XCD-local mode) splits on another XCC
            if (COMB == kCombXcd ? v != mine * (unsigned long long)ns : cnt_total(v) < (unsigned)ns)
                __hip_atomic_store(a.fq.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    if (split >= kTasks) return;
    __syncthreads();
    asm volatile("buffer_inv sc0" ::: "memory");  // workgroup-scope invalidate (the reads are first reads)
    const float *P = a.part + (size_t)s.split0 * 16 * 514;
    for (int t = split;;) {
        comb_task(P, a.fq.ho, a.fq.hos, a.nseq, a.d.HO, b, t >> 1, t & 1, ns, wv, smem);
        t += ns;
        if (t >= kTasks) break;
        __syncthreads();  // the task's LDS is rewritten by the next
        comb_wuv(a.fq.kvb, t >> 1, t & 1, wv);
    }
}

// ONCE: each history row is read by one workgroup (non-temporal loads). FUSE: the launch
// prepares the queries and appends the rows itself (fq_produce; no block launches).
template <bool ONCE, bool FUSE = false, int COMB = kCombNone, bool NORM = false>
__global__ __launch_bounds__(512) void k_attn_q8_mfma(KVL_ATTN_HOT_PARAMS, AttnArgs a) {
    static_assert(COMB == kCombNone || FUSE, "the combine tail is a form of the fused launch");
    KVL_ATTN_HOT_INIT;
    __shared__ __attribute__((aligned(16))) uint8_t smem[kQ8SmemB];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // a fused launch with the projection may have more workgroups than splits (at least
    // kGemvTasks): the ones past the splits only take their projection block. The split count
    // comes in the members argument (-splits; a fused launch is never a block launch), which is
    // preloaded: the argument block's copy would cost every workgroup a memory round trip first.
    if (FUSE && (int)blockIdx.x >= -h.members) {
        fq_gemv<NORM>(a.fq, h.nseq, smem);
        return;
    }
    int b, split, pidx;
    SeqDesc s;
    if (!seq_of<COMB == kCombXcd>(a, h, b, split, pidx, s)) return;
    const int r0 = split * s.rps;
    const int r1 = split == s.nsplit - 1 ? s.len : r0 + s.rps;  // last split takes the rest
    const int nch = (r1 - r0 + kQ8Ch - 1) / kQ8Ch;
    // chunk of this split holding the row appended in this launch, or -1
    const int cpos = FUSE && split == s.nsplit - 1 ? (s.pos - r0) / kQ8Ch : -1;
    if (w >= 4) q8_mix_role<ONCE, FUSE, COMB, NORM>(a, h, s, smem, w - 4, b, r0, r1, nch, pidx, cpos);
    else q8_score_role<FUSE, COMB, NORM>(a, h, s, smem, w, b, r0, r1, nch, pidx, cpos);
    if constexpr (COMB != kCombNone) q8_comb_tail<COMB>(a, s, b, split, smem);
}

bool gemv_fuse_ok(const Dims &d, int B) {
    return B >= 1 && B <= 8 && d.H == 2048 && d.NH == 16 && d.QD == 192 && d.QO == 16 * 192 && d.KVO == 576;
}

bool comb_cross_ok(const SeqTable &t, const Dims &d) {
    if (t.n < 1 || d.NH != 16 || d.R != 512 || d.DN != 128 || d.DV != 128 || d.HO != 16 * 128) return false;
    for (int i = 0; i < t.n; ++i)
        if (t.s[i].nsplit < 16 || t.s[i].nsplit > 255) return false;  // at most two tasks per split
    return true;
}

bool comb_ok(const SeqTable &t, const Dims &d, int total_splits) {
    if (t.n < kXcds || t.n % kXcds != 0 || d.NH != 16 || d.R != 512 || d.DN != 128 || d.DV != 128 ||
        d.HO != 16 * 128)
        return false;
    const int ns = t.s[0].nsplit;
    if (ns < 1 || ns > 255 || ns * t.n != total_splits) return false;  // 255: q8_comb_tail's byte counts
    for (int i = 0; i < t.n; ++i)
        if (t.s[i].nsplit != ns || t.s[i].split0 != i * ns) return false;
    return true;
}

hipError_t launch_attention(hipStream_t st, int kind, int fmt, const SeqTable &t, const Dims &d,
                            int rows_per_split, int total_splits, int lmax,
                            const DecodeWork &w, int members, const FqArgs *fq) {
    AttnArgs a;
    a.fq = fq ? *fq : FqArgs{};
    if (fq && (kind != kAttnQ8Mfma || members > 0 || fmt != kFmtQ8 || d.NH != 16 || d.R != 512 || d.DR != 64 ||
               d.DN != 128 || d.QD != 192 || 17 * t.n > total_splits || !fq->y || !fq->ukt || !fq->cs || !fq->norm ||
               !fq->rows || !fq->flags || !fq->err ||
               (fq->comb == kCombXcd && !comb_ok(t, d, total_splits)) ||
               (fq->comb == kCombCross && !comb_cross_ok(t, d)) || fq->comb < 0 || fq->comb > kCombCross ||
               (fq->comb && (!fq->kvb || !fq->ho || !fq->hos)) || fq->splits != total_splits ||
               (fq->xnorm && (fq->comb != kCombXcd || !fq->gemv)) ||
               (fq->gemv && (!gemv_fuse_ok(d, t.n) || !fq->x || !fq->wq || !fq->wkva ||
                             fq->in != d.H || fq->out0 != d.QO || fq->out1 != d.KVO || (uintptr_t)fq->x % 16 != 0 ||
                             fq->ldx % 4 != 0))))
        return hipErrorInvalidValue;
    a.t = t;
    a.d = d;
    a.part = w.part;
    a.qf = w.qf;
    a.qhi = w.qhi;
    a.qlo = w.qlo;
    a.qs = w.qs;
    a.qrhi = w.qrhi;
    a.qrlo = w.qrlo;
    a.scores = w.scores;
    a.rps = rows_per_split;
    a.lmax = lmax;
    a.smscale = 1.0f / sqrtf((float)d.QD);
    a.members = kind == kAttnGeneric ? 0 : members;
    a.nseq = t.n;
    int grid = total_splits;
    if (fq && fq->gemv) grid = max(grid, kGemvTasks);  // the projection's blocks
    if (a.members > 0) {
        int maxns = 0;
        for (int i = 0; i < t.n; ++i) maxns = max(maxns, t.s[i].nsplit);
        grid = kXcds * t.n * ((maxns + kXcds - 1) / kXcds);
    }
    if (kind == kAttnQ8Mfma) {
        if (a.members > 0) hipLaunchKernelGGL(k_attn_q8_mfma<false>, dim3(grid), dim3(512), 0, st, a.members, a.nseq, a.qhi, a.qlo, a.qrhi, a.qrlo, a.qs, a.qf, a.part, a);
        else if (fq && fq->comb == kCombXcd && fq->gemv && fq->xnorm) hipLaunchKernelGGL((k_attn_q8_mfma<true, true, kCombXcd, true>), dim3(grid), dim3(512), 0, st, -total_splits, a.nseq, a.qhi, a.qlo, a.qrhi, a.qrlo, a.qs, a.qf, a.part, a);
        else if (fq && fq->comb == kCombXcd) hipLaunchKernelGGL((k_attn_q8_mfma<true, true, kCombXcd>), dim3(grid), dim3(512), 0, st, -total_splits, a.nseq, a.qhi, a.qlo, a.qrhi, a.qrlo, a.qs, a.qf, a.part, a);
        else if (fq && fq->comb == kCombCross) hipLaunchKernelGGL((k_attn_q8_mfma<true, true, kCombCross>), dim3(grid), dim3(512), 0, st, -total_splits, a.nseq, a.qhi, a.qlo, a.qrhi, a.qrlo, a.qs, a.qf, a.part, a);
        else if (fq) hipLaunchKernelGGL((k_attn_q8_mfma<true, true>), dim3(grid), dim3(512), 0, st, -total_splits, a.nseq, a.qhi, a.qlo, a.qrhi, a.qrlo, a.qs, a.qf, a.part, a);
        else hipLaunchKernelGGL(k_attn_q8_mfma<true>, dim3(grid), dim3(512), 0, st, a.members, a.nseq, a.qhi, a.qlo, a.qrhi, a.qrlo, a.qs, a.qf, a.part, a);
    } else if (kind == kAttnF32Mfma) {
        if (a.members > 0) hipLaunchKernelGGL(k_attn_f32_mfma<false>, dim3(grid), dim3(256), 0, st, a.members, a.nseq, a.qhi, a.qlo, a.qrhi, a.qrlo, a.qs, a.qf, a.part, a);
        else hipLaunchKernelGGL(k_attn_f32_mfma<true>, dim3(grid), dim3(256), 0, st, a.members, a.nseq, a.qhi, a.qlo, a.qrhi, a.qrlo, a.qs, a.qf, a.part, a);
    } else if (kind == kAttnBF16Mfma) {
        if (a.members > 0) hipLaunchKernelGGL(k_attn_bf16_mfma<false>, dim3(grid), dim3(256), 0, st, a.members, a.nseq, a.qhi, a.qlo, a.qrhi, a.qrlo, a.qs, a.qf, a.part, a);
        else hipLaunchKernelGGL(k_attn_bf16_mfma<true>, dim3(grid), dim3(256), 0, st, a.members, a.nseq, a.qhi, a.qlo, a.qrhi, a.qrlo, a.qs, a.qf, a.part, a);
    } else {
        const int P = fmt == kFmtExp ? t.n * d.NH : t.n;
        if (fmt == kFmtQ8)
            hipLaunchKernelGGL(k_attn_generic<kFmtQ8>, dim3(P), dim3(256), 0, st, a);
        else if (fmt == kFmtF32)
            hipLaunchKernelGGL(k_attn_generic<kFmtF32>, dim3(P), dim3(256), 0, st, a);
        else if (fmt == kFmtBF16)
            hipLaunchKernelGGL(k_attn_generic<kFmtBF16>, dim3(P), dim3(256), 0, st, a);
        else
            hipLaunchKernelGGL(k_attn_generic<kFmtExp>, dim3(P), dim3(256), 0, st, a);
    }
    return hipGetLastError();
}

// ================================================================ combine + W_UV =======

struct CombineArgs {
    SeqTable t;
    Dims d;
    const float *part;
    const uint16_t *kv_b;
    float *mix;
    float *ho;
    uint16_t *hos;
    int fmt;
    int spb;  // k_combine_r512: sequences per block (taken in turn)
};

bool combine_writes_hos(int fmt, const Dims &d) { return fmt != kFmtExp && d.R == 512 && d.DV == 128; }

// One block per (sequence, head). m* = max_s m_s, denom = sum_s l_s e^(m_s - m*),
// mix = sum_s acc_s e^(m_s - m*) / denom; then (compressed formats)
// ho[d] = sum_r kv_b[h*(DN+DV)+DN+d, r] * mix[r] (src/mla_compressed_q8_state.c:239-247).
// Split weights are computed once into LDS; the mix loop issues independent loads.

__global__ __launch_bounds__(256) void k_combine(CombineArgs a) {
    __shared__ float mx[kMaxR];
    __shared__ float wts[kMaxSplits];
    __shared__ float red[256];
    const Dims &d = a.d;
    const int b = blockIdx.x / d.NH, h = blockIdx.x % d.NH, tid = threadIdx.x;
    const SeqDesc &s = a.t.s[b];
    const bool exp = a.fmt == kFmtExp;
    const int G = exp ? 1 : d.NH, DVm = exp ? d.DV : d.R, g = exp ? 0 : h;
    const int sp0 = exp ? b * d.NH + h : s.split0, ns = exp ? 1 : s.nsplit;
    const size_t stride = (size_t)G * (DVm + 2);
    const float *P = a.part + (size_t)sp0 * stride;
    float m = -INFINITY;
    for (int i = tid; i < ns; i += 256) {
        const float mi = P[i * stride + (size_t)G * DVm + g];
        wts[i] = mi;
        m = fmaxf(m, mi);
    }
    red[tid] = m;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) red[tid] = fmaxf(red[tid], red[tid + o]);
        __syncthreads();
    }
    const float M = red[0];
    __syncthreads();
    float den = 0.f;
    for (int i = tid; i < ns; i += 256) {
        const float e = __expf(wts[i] - M);
        wts[i] = e;
        den = fmaf(P[i * stride + (size_t)G * DVm + G + g], e, den);
    }
    red[tid] = den;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) red[tid] += red[tid + o];
        __syncthreads();
    }
    const float inv = 1.0f / red[0];
    float *mixrow = a.mix + ((size_t)b * d.NH + h) * DVm;
    const float *Pg = P + (size_t)g * DVm;
    for (int k = tid; k < DVm; k += 256) {
        float v0 = 0.f, v1 = 0.f, v2 = 0.f, v3 = 0.f;
        int i = 0;
        for (; i + 8 <= ns; i += 8) {
            float p[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) p[q] = Pg[(size_t)(i + q) * stride + k];
            v0 = fmaf(p[0], wts[i], v0);
            v1 = fmaf(p[1], wts[i + 1], v1);
            v2 = fmaf(p[2], wts[i + 2], v2);
            v3 = fmaf(p[3], wts[i + 3], v3);
            v0 = fmaf(p[4], wts[i + 4], v0);
            v1 = fmaf(p[5], wts[i + 5], v1);
            v2 = fmaf(p[6], wts[i + 6], v2);
            v3 = fmaf(p[7], wts[i + 7], v3);
        }
        for (; i < ns; ++i) v0 = fmaf(Pg[(size_t)i * stride + k], wts[i], v0);
        const float v = ((v0 + v1) + (v2 + v3)) * inv;
        mixrow[k] = v;
        if (exp)
            a.ho[(size_t)b * d.HO + (size_t)h * d.DV + k] = v;
        else
            mx[k] = v;
    }
    if (exp) return;
    __syncthreads();
    const int w = tid >> 6, l = tid & 63;
    const uint16_t *wuv = a.kv_b + ((size_t)h * (d.DN + d.DV) + d.DN) * d.R;
    if (d.R == 512 && d.DV == 128) {
        // thread t: output row t/2, latent half t%2 (256 columns streamed as 32 x 16 B)
        const int dd = tid >> 1, half = tid & 1;
        const uint16_t *row = wuv + (size_t)dd * 512 + 256 * half;
        const float *mh = mx + 256 * half;
        float acc0 = 0.f, acc1 = 0.f;
#pragma unroll
        for (int q0 = 0; q0 < 32; q0 += 8) {
            v4i wv[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) wv[q] = *(const v4i *)(row + 8 * (q0 + q));
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const v4f m0 = *(const v4f *)(mh + 8 * (q0 + q));
                const v4f m1 = *(const v4f *)(mh + 8 * (q0 + q) + 4);
                const uint32_t u0 = (uint32_t)wv[q][0], u1 = (uint32_t)wv[q][1];
                const uint32_t u2 = (uint32_t)wv[q][2], u3 = (uint32_t)wv[q][3];
                acc0 = fmaf(__uint_as_float(u0 << 16), m0.x, acc0);
                acc1 = fmaf(__uint_as_float(u0 & 0xffff0000u), m0.y, acc1);
                acc0 = fmaf(__uint_as_float(u1 << 16), m0.z, acc0);
                acc1 = fmaf(__uint_as_float(u1 & 0xffff0000u), m0.w, acc1);
                acc0 = fmaf(__uint_as_float(u2 << 16), m1.x, acc0);
                acc1 = fmaf(__uint_as_float(u2 & 0xffff0000u), m1.y, acc1);
                acc0 = fmaf(__uint_as_float(u3 << 16), m1.z, acc0);
                acc1 = fmaf(__uint_as_float(u3 & 0xffff0000u), m1.w, acc1);
            }
        }
        float acc = acc0 + acc1;
        acc += dpp_f32<0xB1>(acc);  // partner lane t^1 holds the other half
        if (half == 0) a.ho[(size_t)b * d.HO + (size_t)h * d.DV + dd] = acc;
        return;
    }
    for (int dd = w; dd < d.DV; dd += 4) {
        const uint16_t *row = wuv + (size_t)dd * d.R;
        float acc = 0.f;
        for (int r = l; r < d.R; r += 64) acc = fmaf(bf16_to_f32(row[r]), mx[r], acc);
        acc = wave_sum(acc);
        if (l == 0) a.ho[(size_t)b * d.HO + (size_t)h * d.DV + dd] = acc;
    }
}

// Compressed formats with R = 512, DV = 128: the same algebra in one round of memory requests,
// over 2 blocks of 1024 threads per (sequence, head) (twice the blocks of one per head, which
// measured faster than reading each partial once). Block half computes the whole mix and W_UV
// rows [64 half, 64 half + 64) of the head output. Every load is issued up front: wave 0 the
// split maxima and denominators; thread t the partials of latent columns 4 (t % 128) .. +3 for
// the splits s = t / 128 (mod 8), 16 bytes per split (the first kCombPre of them; longer
// histories loop), and its W_UV slice (row t / 16, columns 32 (t % 16) .. + 31). After the
// split weights are in LDS, each thread sums its splits in order, the 8 split groups are added
// in group order through LDS, and 16 lanes per W_UV row reduce its dot product. The head output
// is also written as bf16 hi | lo planes (w.hos), the operand format of launch_gemv_xs. Large
// batches give a block spb sequences of the same (head, half), taken in turn with the W_UV slice
// loaded once, so that the grid stays within one round of the CUs.
// LDS position of mix column c: the 4-column groups of each 32-column row are XOR-permuted by the
// row, so that the W_UV dot's reads (lane q: columns 32 q + 8 c' .. + 7) fall in distinct banks.
constexpr int kCombBlocks = 256;  // k_combine_r512 grid target: one round on the CUs of an MI355X
constexpr int kCombWide = 16;     // k_combine_r512x8: at most this many splits per sequence
__global__ __launch_bounds__(1024) void k_combine_r512(const float *part_, const uint16_t *kv_b_, float *ho_, uint16_t *hos_, int spb_, int nh_, int dn_, int n_, int un_, CombineArgs a) {
    // leading scalar arguments: preloaded into SGPRs at wave start (no argument round trip)
    __shared__ float mx[512];
    __shared__ float wts[kMaxSplits];
    __shared__ v4f red[8][128];
    __shared__ float sinv;
    // un_ > 0: every sequence has un_ splits, sequence b's starting at split b * un_, and the
    // partial loads need no descriptor (one memory round trip less before them)
    DescLane dl{};
    if (un_ == 0) dl = desc_lane(a.t);  // first: the partial loads wait for it
    const int NH = nh_, tid = threadIdx.x;
    // block i takes half i / (grid / 2): both halves of a (sequence, head) run on one XCD
    // (workgroup i on XCD i % 8, NH % 8 == 0), so its split partials, written to memory with
    // non-temporal stores by the attention, come into that XCD's L2 once for the two blocks
    // (the headline stack: 6.34 -> 5.38 us per launch against adjacent halves)
    const int ngh = (int)gridDim.x >> 1, half = (int)blockIdx.x >= ngh;
    const int gh = (int)blockIdx.x - half * ngh, grp = gh / NH, h = gh % NH;
    const int dd = 64 * half + (tid >> 4), q = tid & 15;
    const uint16_t *row = kv_b_ + ((size_t)h * (dn_ + 128) + dn_ + dd) * 512 + 32 * q;
    v4i wv[4];  // held for every sequence of the block
#pragma unroll
    for (int c = 0; c < 4; ++c) wv[c] = *(const v4i *)(row + 8 * c);
    // split group: uniform within a wave (128-thread groups)
    const int sg = __builtin_amdgcn_readfirstlane(tid >> 7);
    const size_t stride = (size_t)NH * (512 + 2);
    const int b_end = min((grp + 1) * spb_, n_);
    for (int b = grp * spb_; b < b_end; ++b) {
        // column group of this thread, opaque to the compiler so that the per-split addresses
        // below are formed in each iteration instead of being held (spilled) across the loop
        int c4 = tid & 127;
        asm volatile("" : "+v"(c4));
        const int ns = un_ > 0 ? un_ : lane_pick(dl.nsplit, b);
        const float *P = part_ + (size_t)(un_ > 0 ? b * un_ : lane_pick(dl.split0, b)) * stride;
        const float *Pm = P + (size_t)NH * 512 + h;  // split i: m at Pm[i * stride], l at + NH
        float m0 = 0.f, l0 = 0.f;
        if (tid < 64) {
            const int i0 = min(tid, ns - 1);
            m0 = Pm[(size_t)i0 * stride];
            l0 = Pm[(size_t)i0 * stride + NH];
        }
        const float *Pg = P + (size_t)h * 512 + 4 * c4;
        v4f pre[kCombPre];
#pragma unroll
        for (int i = 0; i < kCombPre; ++i)  // sg is uniform within a wave: splits past ns are not loaded
            pre[i] = sg + 8 * i < ns ? *(const v4f *)(Pg + (size_t)(sg + 8 * i) * stride) : v4f{0.f, 0.f, 0.f, 0.f};
        if (tid < 64) {
            float m = tid < ns ? m0 : -INFINITY;
            for (int i = tid + 64; i < ns; i += 64) m = fmaxf(m, Pm[(size_t)i * stride]);
            m = wave_max(m);
            float den = 0.f;
            if (tid < ns) {
                const float e = __expf(m0 - m);
                wts[tid] = e;
                den = l0 * e;
            }
            for (int i = tid + 64; i < ns; i += 64) {
                const float e = __expf(Pm[(size_t)i * stride] - m);
                wts[i] = e;
                den = fmaf(Pm[(size_t)i * stride + NH], e, den);
            }
            den = wave_sum(den);
            if (tid == 0) sinv = 1.0f / den;
        }
        __syncthreads();
        v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kCombPre; ++i) {
            const int sp = sg + 8 * i;
            if (sp < ns) {
                const float wt = wts[sp];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = fmaf(pre[i][e], wt, acc[e]);
            }
        }
        for (int sp = sg + 8 * kCombPre; sp < ns; sp += 8 * kCombPre) {
            v4f more[kCombPre];
#pragma unroll
            for (int i = 0; i < kCombPre; ++i)
                more[i] = sp + 8 * i < ns ? *(const v4f *)(Pg + (size_t)(sp + 8 * i) * stride) : v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < kCombPre; ++i) {
                if (sp + 8 * i < ns) {
                    const float wt = wts[sp + 8 * i];
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[e] = fmaf(more[i][e], wt, acc[e]);
                }
            }
        }
        red[sg][c4] = acc;
        __syncthreads();
        if (tid < 512) {
            const int cq = tid >> 2, e = tid & 3;
            float v = red[0][cq][e];
#pragma unroll
            for (int g8 = 1; g8 < 8; ++g8) v += red[g8][cq][e];
            mx[mx_pos(tid)] = v * sinv;
        }
        __syncthreads();
        float acc0 = 0.f, acc1 = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const v4f m0v = *(const v4f *)(mx + mx_pos(32 * q + 8 * c));
            const v4f m1v = *(const v4f *)(mx + mx_pos(32 * q + 8 * c + 4));
            const uint32_t u0 = (uint32_t)wv[c][0], u1 = (uint32_t)wv[c][1];
            const uint32_t u2 = (uint32_t)wv[c][2], u3 = (uint32_t)wv[c][3];
            acc0 = fmaf(__uint_as_float(u0 << 16), m0v.x, acc0);
            acc1 = fmaf(__uint_as_float(u0 & 0xffff0000u), m0v.y, acc1);
            acc0 = fmaf(__uint_as_float(u1 << 16), m0v.z, acc0);
            acc1 = fmaf(__uint_as_float(u1 & 0xffff0000u), m0v.w, acc1);
            acc0 = fmaf(__uint_as_float(u2 << 16), m1v.x, acc0);
            acc1 = fmaf(__uint_as_float(u2 & 0xffff0000u), m1v.y, acc1);
            acc0 = fmaf(__uint_as_float(u3 << 16), m1v.z, acc0);
            acc1 = fmaf(__uint_as_float(u3 & 0xffff0000u), m1v.w, acc1);
        }
        const float hsum = row16_sum(acc0 + acc1);  // the 16 lanes of row dd
        if (q == 0) {
            const size_t o = (size_t)b * a.d.HO + (size_t)h * 128 + dd;
            ho_[o] = hsum;
            uint16_t hi, lo;
            split_bf16(hsum, hi, lo);
            hos_[o] = hi;
            hos_[(size_t)n_ * a.d.HO + o] = lo;
        }
        __syncthreads();  // wts, red and mx are rewritten for the next sequence
    }
}

// The same combine for 8 sequences of one (head, half) per block, for large batches: the 128
// threads of sequence j (waves 2j, 2j+1) merge its splits -- wave 2j computes the split maxima,
// weights and denominator exactly as wave 0 of k_combine_r512 does, and thread (j, c) forms
// each split group's sum of columns 4c .. 4c+3 and adds the eight group sums in group order,
// the operations k_combine_r512 spreads over its threads -- then every thread takes its W_UV row
// slice through the eight mixes. The outputs equal k_combine_r512's bit for bit, with W_UV read
// once per 8 sequences and 8 times fewer blocks.
__global__ __launch_bounds__(1024) void k_combine_r512x8(const float *part_, const uint16_t *kv_b_, float *ho_, uint16_t *hos_, int spb_, int nh_, int dn_, int n_, CombineArgs a) {
    // leading scalar arguments: preloaded into SGPRs at wave start (no argument round trip)
    __shared__ float mx[8][512];
    __shared__ float wts[8][kCombWide];
    __shared__ float sinv[8];
    const DescLane dl = desc_lane(a.t);  // first: the partial loads wait for it
    const int NH = nh_, tid = threadIdx.x;
    // halves on one XCD, as in k_combine_r512 (ragged 64-sequence legs: 15.6 -> 14.3 us)
    const int ngh = (int)gridDim.x >> 1, half = (int)blockIdx.x >= ngh;
    const int gh = (int)blockIdx.x - half * ngh, grp = gh / NH, h = gh % NH;
    const int dd = 64 * half + (tid >> 4), q = tid & 15;
    const uint16_t *row = kv_b_ + ((size_t)h * (dn_ + 128) + dn_ + dd) * 512 + 32 * q;
    v4i wv[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) wv[c] = *(const v4i *)(row + 8 * c);
    const int j = __builtin_amdgcn_readfirstlane(tid >> 7), c4 = tid & 127, lw = tid & 127;
    const int b = grp * 8 + j;
    const bool live = b < n_;
    const size_t stride = (size_t)NH * (512 + 2);
    const int ns = live ? lane_pick(dl.nsplit, b) : 0;
    const float *P = part_ + (size_t)lane_pick(dl.split0, live ? b : 0) * stride;
    const float *Pm = P + (size_t)NH * 512 + h;
    const float *Pg = P + (size_t)h * 512 + 4 * c4;
    v4f pre[kCombWide];
#pragma unroll
    for (int i = 0; i < kCombWide; ++i)
        pre[i] = i < ns ? *(const v4f *)(Pg + (size_t)i * stride) : v4f{0.f, 0.f, 0.f, 0.f};
    if (lw < 64 && live) {
        const float m0 = Pm[(size_t)min(lw, ns - 1) * stride];
        const float l0 = Pm[(size_t)min(lw, ns - 1) * stride + NH];
        float m = lw < ns ? m0 : -INFINITY;
        m = wave_max(m);
        float den = 0.f;
        if (lw < ns) {
            const float e = __expf(m0 - m);
            wts[j][lw] = e;
            den = l0 * e;
        }
        den = wave_sum(den);
        if (lw == 0) sinv[j] = 1.0f / den;
    }
    __syncthreads();
    if (live) {
        // split group g8 holds splits g8, g8 + 8, ...; the groups are added in order
        v4f v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int g8 = 0; g8 < 8; ++g8) {
            v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = g8; i < kCombWide; i += 8) {
                if (i < ns) {
                    const float wt = wts[j][i];
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[e] = fmaf(pre[i][e], wt, acc[e]);
                }
            }
            if (g8 == 0) v = acc;
            else v += acc;
        }
        *(v4f *)(&mx[j][mx_pos(4 * c4)]) = v * sinv[j];
    }
    __syncthreads();
#pragma unroll 1
    for (int jj = 0; jj < 8 && grp * 8 + jj < n_; ++jj) {
        const float *mh = mx[jj];
        float acc0 = 0.f, acc1 = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const v4f m0v = *(const v4f *)(mh + mx_pos(32 * q + 8 * c));
            const v4f m1v = *(const v4f *)(mh + mx_pos(32 * q + 8 * c + 4));
            const uint32_t u0 = (uint32_t)wv[c][0], u1 = (uint32_t)wv[c][1];
            const uint32_t u2 = (uint32_t)wv[c][2], u3 = (uint32_t)wv[c][3];
            acc0 = fmaf(__uint_as_float(u0 << 16), m0v.x, acc0);
            acc1 = fmaf(__uint_as_float(u0 & 0xffff0000u), m0v.y, acc1);
            acc0 = fmaf(__uint_as_float(u1 << 16), m0v.z, acc0);
            acc1 = fmaf(__uint_as_float(u1 & 0xffff0000u), m0v.w, acc1);
            acc0 = fmaf(__uint_as_float(u2 << 16), m1v.x, acc0);
            acc1 = fmaf(__uint_as_float(u2 & 0xffff0000u), m1v.y, acc1);
            acc0 = fmaf(__uint_as_float(u3 << 16), m1v.z, acc0);
            acc1 = fmaf(__uint_as_float(u3 & 0xffff0000u), m1v.w, acc1);
        }
        const float hsum = row16_sum(acc0 + acc1);
        if (q == 0) {
            const size_t o = (size_t)(grp * 8 + jj) * a.d.HO + (size_t)h * 128 + dd;
            ho_[o] = hsum;
            uint16_t hi, lo;
            split_bf16(hsum, hi, lo);
            hos_[o] = hi;
            hos_[(size_t)n_ * a.d.HO + o] = lo;
        }
    }
}

hipError_t launch_combine(hipStream_t st, int fmt, const SeqTable &t, const Dims &d,
                          const uint16_t *kv_b, const DecodeWork &w) {
    if (d.R > kMaxR) return hipErrorInvalidValue;
    CombineArgs a{t, d, w.part, kv_b, w.mix, w.ho, w.hos, fmt, 1};
    int maxns = 0, un = t.n > 0 ? t.s[0].nsplit : 0;
    for (int i = 0; i < t.n; ++i) {
        maxns = max(maxns, t.s[i].nsplit);
        if (t.s[i].nsplit != un || t.s[i].split0 != i * un) un = 0;
    }
    if (combine_writes_hos(fmt, d) && t.n >= 32 && maxns <= kCombWide) {
        hipLaunchKernelGGL(k_combine_r512x8, dim3(2 * ((t.n + 7) / 8) * d.NH), dim3(1024), 0, st, a.part, a.kv_b, a.ho, a.hos, a.spb, d.NH, d.DN, t.n, a);
    } else if (combine_writes_hos(fmt, d)) {
        // up to kCombBlocks blocks; a block takes spb sequences of one (head, half) in turn
        a.spb = max(1, (2 * t.n * d.NH + kCombBlocks - 1) / kCombBlocks);
        const int groups = (t.n + a.spb - 1) / a.spb;
        hipLaunchKernelGGL(k_combine_r512, dim3(2 * groups * d.NH), dim3(1024), 0, st, a.part, a.kv_b, a.ho, a.hos, a.spb, d.NH, d.DN, t.n, un, a);
    } else {
        hipLaunchKernelGGL(k_combine, dim3(t.n * d.NH), dim3(256), 0, st, a);
    }
    return hipGetLastError();
}

// ================================================================ copy =================

__global__ __launch_bounds__(256) void k_copy(v4i *dst, const v4i *src, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        dst[i] = src[i];
}

// Streaming read of n 16-byte words, folded by XOR; the fold reaches memory only for one
// (practically never occurring) pattern, which keeps every load live: a read-bandwidth probe.
// Each block streams a contiguous 1/gridDim of the buffer with 8 non-temporal loads of 16 bytes
// in flight per thread: contiguous per-block ranges reached 6.2-6.3 TB/s on MI355X, a
// grid-stride order over the same bytes 5.1-5.5 TB/s (plain loads; non-temporal ones, as the
// decode's history streams use, 5-10 % more in a grid-stride order).
__global__ __launch_bounds__(256) void k_read(const v4i *src, size_t n, v4i *sink) {
    const size_t per = (n + gridDim.x - 1) / gridDim.x;
    const size_t b0 = (size_t)blockIdx.x * per, b1 = b0 + per < n ? b0 + per : n;
    v4i acc = {0, 0, 0, 0};
    size_t i = b0 + threadIdx.x;
    for (; i + 7 * 256 < b1; i += 8 * 256) {
        v4i v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = __builtin_nontemporal_load(src + i + 256 * u);
#pragma unroll
        for (int u = 0; u < 8; ++u) acc ^= v[u];
    }
    for (; i < b1; i += 256) acc ^= __builtin_nontemporal_load(src + i);
    if ((acc.x ^ acc.y ^ acc.z ^ acc.w) == 0x5a17c3e1) sink[(size_t)blockIdx.x * 256 + threadIdx.x] = acc;
}

hipError_t launch_read(hipStream_t st, const void *src, size_t bytes, void *sink) {
    const size_t n = bytes / 16;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_read, dim3(kReadBlocks), dim3(256), 0, st, (const v4i *)src, n, (v4i *)sink);
    return hipGetLastError();
}

// Launch-cost probe: a kernel whose workgroups do nothing.
__global__ __launch_bounds__(1024) void k_empty() {}

hipError_t launch_empty(hipStream_t st) {
    hipLaunchKernelGGL(k_empty, dim3(256), dim3(1024), 0, st);
    return hipGetLastError();
}

hipError_t launch_copy(hipStream_t st, void *dst, const void *src, size_t bytes) {
    const size_t n = bytes / 16;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_copy, dim3(4096), dim3(256), 0, st, (v4i *)dst, (const v4i *)src, n);
    return hipGetLastError();
}

// ================================================================ synthetic history ====

struct FillArgs {
    void *a, *b, *c;
    int R, DR, row0, nrows, fmt;
    uint64_t seed;
};

// One wave per row. Element e of global row j draws synth_normal(seed, j*(R+DR) + e).
// Q8: the R latents go through the history quantiser, the DR RoPE values are rounded to
// bf16. F32: all values are rounded to bf16 first (bf16-representable fp32 history). BF16:
// the same bf16 values, stored as bf16 (a BF16 and an F32 history of one seed hold equal rows).
__global__ __launch_bounds__(256) void k_fill_history(FillArgs a) {
    const int wv = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, l = threadIdx.x & 63;
    if (wv >= a.nrows) return;
    const int j = a.row0 + wv;
    const uint64_t base = (uint64_t)j * (uint64_t)(a.R + a.DR);
    if (a.fmt == kFmtQ8) {
        float m = 0.f;
        for (int e = l; e < a.R; e += 64) m = fmaxf(m, fabsf(synth_normal(a.seed, base + e)));
        m = wave_max(m);
        const bool zero = !(m > 0.0f) || !isfinite(m);
        const float scale = zero ? 1.0f : m / 127.0f;
        const float inv = zero ? 0.0f : 1.0f / scale;
        int8_t *codes = (int8_t *)a.a + (size_t)j * a.R;
        for (int e = l; e < a.R; e += 64) {
            float v = roundf(synth_normal(a.seed, base + e) * inv);
            v = fminf(fmaxf(v, -127.f), 127.f);
            codes[e] = zero ? (int8_t)0 : (int8_t)v;
        }
        if (l == 0) ((float *)a.b)[j] = scale;
        uint16_t *rope = (uint16_t *)a.c + (size_t)j * a.DR;
        for (int e = l; e < a.DR; e += 64) rope[e] = f32_to_bf16_rne(synth_normal(a.seed, base + a.R + e));
    } else if (a.fmt == kFmtBF16) {
        uint16_t *lat = (uint16_t *)a.a + (size_t)j * a.R;
        uint16_t *rope = (uint16_t *)a.b + (size_t)j * a.DR;
        for (int e = l; e < a.R; e += 64) lat[e] = f32_to_bf16_rne(synth_normal(a.seed, base + e));
        for (int e = l; e < a.DR; e += 64) rope[e] = f32_to_bf16_rne(synth_normal(a.seed, base + a.R + e));
    } else {
        float *lat = (float *)a.a + (size_t)j * a.R;
        float *rope = (float *)a.b + (size_t)j * a.DR;
        for (int e = l; e < a.R; e += 64) lat[e] = bf16_to_f32(f32_to_bf16_rne(synth_normal(a.seed, base + e)));
        for (int e = l; e < a.DR; e += 64)
            rope[e] = bf16_to_f32(f32_to_bf16_rne(synth_normal(a.seed, base + a.R + e)));
    }
}

hipError_t launch_fill_history(hipStream_t st, int fmt, void *a, void *b, void *c, int R,
                               int DR, int row0, int nrows, uint64_t seed) {
    if (nrows <= 0) return hipSuccess;
    FillArgs f{a, b, c, R, DR, row0, nrows, fmt, seed};
    hipLaunchKernelGGL(k_fill_history, dim3((nrows + 3) / 4), dim3(256), 0, st, f);
    return hipGetLastError();
}

}  // namespace kvl
