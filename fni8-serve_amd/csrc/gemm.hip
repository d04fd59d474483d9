// int8 x int8 -> int32 GEMM with the fused dequant epilogue (gfx950).
//
//   y[m, n] = fp16(((float)sum_k a[m, k] * w[n, k]) * as[m] * ws[n] (+ bias[n]))
//
// Both operands are K-contiguous (the per_row_i8 weight is [N, K] row-major),
// which is exactly the per-lane layout of v_mfma_i32_16x16x64_i8: every lane
// feeds 16 consecutive int8 of one row of A and of one row of B, so neither
// operand needs a transpose anywhere.
//
// This file holds the skinny kernel (a dense and a grouped, expert segment,
// form) for what the 128-byte slabs of decode_mfma.hip do not take at M <= 64
// and in small expert segments: any K % 4 == 0, rows 4-byte aligned.  HBM-bound
// weight streaming: a workgroup owns 16 * NB weight rows, its waves split K,
// every lane streams 16-byte loads of W straight into MFMA operands (no LDS
// staging: each weight byte is used once), partial sums are reduced across
// waves through LDS, then the epilogue.  It also picks the kernel of every GEMM.
// Integer accumulation is exact, so every kernel (and any split of K) gives
// bit-identical accumulators.
#include "common.h"

namespace {

using fni8::mfma_i8;

__device__ __forceinline__ i32x4 ld16(const int8_t* p) {
    return *reinterpret_cast<const fni8::i32x4_a4*>(p);
}

// Streaming load: non-temporal hint, for data read exactly once.
__device__ __forceinline__ i32x4 ld16_stream(const int8_t* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const fni8::i32x4_a4*>(p));
}

// ---------------------------------------------------------------------------
// skinny kernel
// ---------------------------------------------------------------------------
// MT: 16-row blocks of activations (M <= 16 * MT); NB: 16-row blocks of weight
// rows per workgroup (every wave streams all NB blocks over its K share, so
// each activation fragment feeds NB MFMAs); WAVES: waves splitting K;
// U: 64-byte K units per loop trip (U * NB 16-byte weight loads in flight per
// lane).  Weight loads are non-temporal: each byte is used once, so they are
// kept from displacing the activations in L2.  The last K % 64 bytes are one
// more unit, taken by the last wave with zeros past the row's end.
template <int MT, int NB, int WAVES, int U, bool GROUPED>
__global__ __launch_bounds__(WAVES * 64) void gemm_skinny_kernel(
    const int8_t* __restrict__ aq, int64_t lda, const float* __restrict__ as,
    const int32_t* __restrict__ row_index, int M, int K, const int8_t* __restrict__ w,
    const float* __restrict__ ws, int N, int E, const int32_t* __restrict__ seg_off,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ y, int64_t ldy,
    int32_t* __restrict__ acc_out) {
    constexpr int BM = 16 * MT;
    constexpr int BN = 16 * NB;
    __shared__ i32x4 red[WAVES][MT * NB][64];

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    // dense: x = n-tile, y = m-tile; grouped: x = segment tile slot, y = n-tile
    const int nt = GROUPED ? blockIdx.y : blockIdx.x;

    int m0, m1;
    const int8_t* wexp = w;
    const float* wsexp = ws;
    const uint16_t* bexp = bias;
    if constexpr (GROUPED) {
        int e;
        if (!fni8::find_group_tile(seg_off, E, BM, blockIdx.x, M, e, m0, m1)) return;
        wexp += (int64_t)e * N * K;
        wsexp += (int64_t)e * N;
        if (bias) bexp += (int64_t)e * N;
    } else {
        m0 = blockIdx.y * BM;
        m1 = min(M, m0 + BM);
    }

    const int r = lane & 15, g = lane >> 4;
    const int8_t* wrow[NB];
    bool nvalid[NB];
    float wsc[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int n = nt * BN + b * 16 + r;
        nvalid[b] = n < N;
        wrow[b] = wexp + (int64_t)(nvalid[b] ? n : 0) * K + g * 16;
        wsc[b] = nvalid[b] ? wsexp[n] : 0.f;  // epilogue scale, fetched early
    }
    const int8_t* arow[MT];
    bool avalid[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int mr = m0 + mt * 16 + r;
        avalid[mt] = mr < m1;
        int src = mr;
        if (GROUPED && row_index != nullptr && avalid[mt]) src = row_index[mr];
        arow[mt] = aq + (int64_t)(avalid[mt] ? src : 0) * lda + g * 16;
    }

    const int units = K >> 6;
    const int per = (units + WAVES - 1) / WAVES;
    const int u0 = wave * per;
    const int u1 = min(units, u0 + per);

    i32x4 acc[MT][NB];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[mt][b] = i32x4{0, 0, 0, 0};

    for (int u = u0; u < u1; u += U) {
        i32x4 bw[NB][U];
        i32x4 ax[MT][U];
#pragma unroll
        for (int j = 0; j < U; j++) {
            const bool ok = (u + j) < u1;
#pragma unroll
            for (int b = 0; b < NB; b++)
                bw[b][j] = (ok && nvalid[b]) ? ld16_stream(wrow[b] + (int64_t)(u + j) * 64)
                                             : i32x4{0, 0, 0, 0};
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
                ax[mt][j] = (ok && avalid[mt]) ? ld16(arow[mt] + (int64_t)(u + j) * 64)
                                               : i32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (int j = 0; j < U; j++)
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) acc[mt][b] = mfma_i8(ax[mt][j], bw[b][j], acc[mt][b]);
    }

    if ((K & 63) != 0 && wave == WAVES - 1) {
        const int kt = units * 64 + g * 16;
        i32x4 bt[NB], at[MT];
#pragma unroll
        for (int b = 0; b < NB; b++) bt[b] = fni8::ld16_tail(wrow[b] - g * 16, kt, K);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) at[mt] = fni8::ld16_tail(arow[mt] - g * 16, kt, K);
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) acc[mt][b] = mfma_i8(at[mt], bt[b], acc[mt][b]);
    }

#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int b = 0; b < NB; b++) red[wave][mt * NB + b][lane] = acc[mt][b];
    __syncthreads();

    // Each (m-block, n-block) result is summed over the waves by one wave-sized
    // group of threads; a thread keeps the lane layout of the MFMA result.
    for (int idx = threadIdx.x; idx < MT * NB * 64; idx += WAVES * 64) {
        const int mb = idx >> 6, ln = idx & 63;
        const int mt = mb / NB, b = mb % NB;
        i32x4 s = red[0][mb][ln];
#pragma unroll
        for (int wv = 1; wv < WAVES; wv++) s += red[wv][mb][ln];
        const int col = nt * BN + b * 16 + (ln & 15);
        if (col >= N) continue;
        // ln == lane (the stride is a whole number of waves), so wsc[b] is this
        // column's scale.
        const float wscale = wsc[b];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int mr = m0 + mt * 16 + (ln >> 4) * 4 + i;
            if (mr >= m1) continue;
            int src = mr;
            if (GROUPED && row_index != nullptr) src = row_index[mr];
            y[(int64_t)mr * ldy + col] = fni8::dequant_one(s[i], as[src], wscale, bexp, col);
            if (acc_out) acc_out[(int64_t)mr * N + col] = s[i];
        }
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
struct Args {
    const int8_t* aq;
    int64_t lda;
    const float* as;
    const int32_t* row_index;
    int M, K;
    const int8_t* w;
    const float* ws;
    int N, E;
    const int32_t* seg_off;
    const uint16_t* bias;
    uint16_t* y;
    int64_t ldy;
    int32_t* acc_out;
};

template <int MT, int NB, int WAVES, int U, bool GROUPED>
void launch_skinny(const Args& a, unsigned mslots, hipStream_t st) {
    const unsigned ntn = (unsigned)((a.N + 16 * NB - 1) / (16 * NB));
    dim3 grid = GROUPED ? dim3(mslots, ntn) : dim3(ntn, mslots), block(WAVES * 64);
    hipLaunchKernelGGL((gemm_skinny_kernel<MT, NB, WAVES, U, GROUPED>), grid, block, 0, st,
                       a.aq, a.lda, a.as, a.row_index, a.M, a.K, a.w, a.ws, a.N, a.E,
                       a.seg_off, a.bias, a.y, a.ldy, a.acc_out);
}

// M <= 64 tokens, K not a multiple of 128 (a shard's width) or unaligned rows
// (N x K = 2080 x 5472, whose last 32 bytes are the tail unit: 7.4 us at one token,
// 12.5 at 24; one dot4 output per lane took 270 and 236).
// Launch shapes chosen by measurement on MI355X (weights streamed from HBM): 4-wave groups with 16 loads in flight per lane for K = 4096, 8 waves x 4
// loads for long K; two weight blocks per wave once M >= 16 on wide N so each
// activation fragment is reused.
void launch_decode(const Args& a, hipStream_t st) {
    const int M = a.M, N = a.N, K = a.K;
    const bool wide = N >= 16384, longk = K >= 8192, mid = N >= 6144;
    if (M <= 4) {
        if (longk) launch_skinny<1, 1, 8, 4, false>(a, 1, st);
        else launch_skinny<1, 1, 4, 16, false>(a, 1, st);
    } else if (M <= 16) {
        if (wide) launch_skinny<1, 2, 2, 16, false>(a, 1, st);
        else if (longk) launch_skinny<1, 1, 16, 4, false>(a, 1, st);
        else if (mid) launch_skinny<1, 2, 2, 16, false>(a, 1, st);
        else launch_skinny<1, 1, 4, 16, false>(a, 1, st);
    } else if (M <= 32) {
        if (wide || (mid && !longk)) launch_skinny<2, 2, 4, 8, false>(a, 1, st);
        else if (longk) launch_skinny<2, 1, 16, 4, false>(a, 1, st);
        else launch_skinny<2, 1, 4, 16, false>(a, 1, st);
    } else {
        if (wide) launch_skinny<4, 2, 4, 4, false>(a, 1, st);
        else if (longk) launch_skinny<4, 1, 8, 4, false>(a, 1, st);
        else if (mid) launch_skinny<4, 2, 8, 2, false>(a, 1, st);
        else launch_skinny<4, 1, 4, 8, false>(a, 1, st);
    }
}

}  // namespace

namespace fni8h {

int launch_gemm(const int8_t* aq, int64_t lda, const float* as, const int32_t* row_index,
                int64_t M, int64_t K, const int8_t* w, const float* ws, int64_t N,
                int64_t E, const int32_t* seg_off, const uint16_t* bias, uint16_t* y,
                int64_t ldy, int32_t* acc_out, hipStream_t st, int8_t* work,
                int64_t work_bytes) {
    if (M == 0) return FNI8_OK;
    Args a{aq, lda, as, row_index, (int)M, (int)K, w, ws, (int)N, (int)E, seg_off, bias, y,
           ldy, acc_out};
    const bool grouped = E > 0;
    int rc = FNI8_OK;
    if (grouped) {
        // Expert segments: average rows per expert picks the kernel -- the MFMA
        // decode kernel in grouped form up to 4 rows per expert (the skinny
        // kernel where it does not take the shape), the tile kernel above.
        const double avg = (double)M / (double)E;
        if (avg <= 4.0) {
            rc = launch_decode_mfma_grouped(aq, lda, as, row_index, M, K, w, ws, E, N, seg_off,
                                            bias, y, ldy, acc_out, st);
            if (rc == 1) {
                rc = FNI8_OK;
                const unsigned slots = (unsigned)((M + 15) / 16 + E);
                if (K >= 1024) launch_skinny<1, 1, 4, 8, true>(a, slots, st);
                else launch_skinny<1, 1, 2, 8, true>(a, slots, st);
            }
        } else {
            rc = launch_tile32(aq, lda, as, row_index, M, K, w, ws, N, E, seg_off, bias, y, ldy,
                               acc_out, st);
        }
    } else if (M <= 64) {
        rc = launch_decode_q(aq, lda, as, M, K, w, ws, N, bias, y, ldy, acc_out, st);
        if (rc == 1) rc = launch_decode_mfma(aq, lda, as, M, K, w, ws, N, bias, y, ldy, acc_out, st);
        if (rc == 1) {
            rc = FNI8_OK;
            launch_decode(a, st);
        }
    } else {
        rc = launch_pp(aq, lda, as, M, K, w, ws, N, bias, y, ldy, acc_out, work, work_bytes, st);
        if (rc == 1)
            rc = launch_tile32(aq, lda, as, row_index, M, K, w, ws, N, 0, seg_off, bias, y, ldy,
                               acc_out, st);
    }
    if (rc) return rc;
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error_detail("gemm launch: %s", hipGetErrorString(e));
        return FNI8_ERR_LAUNCH;
    }
    return FNI8_OK;
}

}  // namespace fni8h
