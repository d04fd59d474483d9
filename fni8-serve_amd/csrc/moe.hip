// MoE routing sort and weighted combine (gfx950).
//
// sort:    one workgroup per expert, its waves owning contiguous runs of the T*k
//          ids.  Pass 1 counts the ids below and equal to the expert (one block
//          exchange) -> the segment start and each wave's first row, with no
//          global atomics.  Pass 2 places the wave's entries in id order (the
//          rank inside 256 ids from four ballots), so the segment keeps the
//          (token, slot) order of `(topi == e).nonzero()` -- a deterministic,
//          stable counting sort.  Up to 1024 ids a wave stay in registers
//          between the passes.
// combine: one workgroup per token; each lane owns 8 consecutive hidden
//          elements and sums the token's expert rows in ascending expert id
//          with fp16 rounding after every product and add, matching the
//          sequential index_add_ of the per-expert loop.
#include "common.h"

namespace {

constexpr int kMaxTopK = 32;

// Bound by latency: every workgroup reads all ids (from L2) and meets once.
// Walking 1024 ids at a time with two block barriers each took 48 us for 24000
// ids and 128 experts on MI355X; this takes 8.3 (16 waves).
// KEEP: steps held in registers; each costs its share of the start, so as few as
// the ids of a launch need.
template <int WAVES, int KEEP>
__global__ __launch_bounds__(WAVES * 64) void moe_sort_kernel(
    const int32_t* __restrict__ topi, int Tk, int k, int E, int32_t* __restrict__ seg_off,
    int32_t* __restrict__ row_token, int32_t* __restrict__ pos) {
    constexpr int STEP = 256;  // ids per wave and step, four per lane
    __shared__ int lds[2][WAVES];
    const int e = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int steps = (Tk - 1) / (STEP * WAVES) + 1;  // rounded up; no sum here passes 2^31
    const int64_t first = (int64_t)wave * steps * STEP + lane * 4;

    // ids i .. i+3 (-1 past the end)
    auto load = [&](int s) {
        const int64_t i = first + (int64_t)s * STEP;
        i32x4 v = {-1, -1, -1, -1};
        if (i + 3 < Tk) {
            v = *reinterpret_cast<const fni8::i32x4_a4*>(topi + i);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (i + j < Tk) v[j] = topi[i + j];
        }
        return v;
    };
    int lt = 0, eq = 0;
    auto count = [&](i32x4 v) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            lt += (v[j] >= 0 && v[j] < e) ? 1 : 0;
            eq += v[j] == e ? 1 : 0;
        }
    };
    i32x4 kept[KEEP];
#pragma unroll
    for (int s = 0; s < KEEP; s++) kept[s] = s < steps ? load(s) : i32x4{-1, -1, -1, -1};
#pragma unroll
    for (int s = 0; s < KEEP; s++) count(kept[s]);
    for (int s = KEEP; s < steps; s++) count(load(s));
    lt = fni8::wave_sum_i32(lt);
    eq = fni8::wave_sum_i32(eq);
    if (lane == 0) {
        lds[0][wave] = lt;
        lds[1][wave] = eq;
    }
    __syncthreads();
    int start = 0, total = 0, before = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {
        start += lds[0][w];
        total += lds[1][w];
        before += w < wave ? lds[1][w] : 0;
    }
    if (threadIdx.x == 0) {
        seg_off[e] = start;
        if (e == E - 1) seg_off[E] = start + total;
    }

    int base = start + before;
    const uint64_t below = ((uint64_t)1 << lane) - 1;  // the lanes before this one
    auto place = [&](i32x4 v, int s) {
        const int64_t i = first + (int64_t)s * STEP;
        if (e == 0) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (i + j < Tk && (v[j] < 0 || v[j] >= E)) pos[i + j] = -1;  // no row
        }
        uint64_t hit[4];
        int p = base, n = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            hit[j] = __ballot(v[j] == e);
            p += __builtin_popcountll(hit[j] & below);
            n += __builtin_popcountll(hit[j]);
        }
        if (n == 0) return;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (v[j] == e) {
                row_token[p] = (int)((uint32_t)(i + j) / (uint32_t)k);
                pos[i + j] = p;
                p++;
            }
        }
        base += n;
    };
#pragma unroll
    for (int s = 0; s < KEEP; s++)
        if (s < steps) place(kept[s], s);
    for (int s = KEEP; s < steps; s++) place(load(s), s);
}

// Combine for k <= KM (the common top-8): the slots are sorted by expert id
// with an odd-even transposition network (static register indices, stable, so
// the order is that of the insertion sort below), all k rows of the token are
// loaded up front, then summed in that order with the same fp16 roundings.
template <int KM>
__global__ __launch_bounds__(256) void moe_combine_small_kernel(
    const uint16_t* __restrict__ yr, int H, const int32_t* __restrict__ topi,
    const uint16_t* __restrict__ topw, const int32_t* __restrict__ pos, int k,
    int Tk, uint16_t* __restrict__ out) {
    const int t = blockIdx.x;
    int eid[KM], ord[KM];
#pragma unroll
    for (int j = 0; j < KM; j++) {
        eid[j] = j < k ? topi[(int64_t)t * k + j] : 0x7fffffff;
        ord[j] = j;
    }
#pragma unroll
    for (int r = 0; r < KM; r++)
#pragma unroll
        for (int a = r & 1; a + 1 < KM; a += 2)
            if (eid[a] > eid[a + 1]) {
                const int e0 = eid[a], o0 = ord[a];
                eid[a] = eid[a + 1];
                ord[a] = ord[a + 1];
                eid[a + 1] = e0;
                ord[a + 1] = o0;
            }
    int64_t row[KM];
    float wgt[KM];
    bool ok[KM];
#pragma unroll
    for (int j = 0; j < KM; j++) {
        ok[j] = false;
        row[j] = 0;
        wgt[j] = 0.f;
        if (j < k) {
            const int slot = ord[j];
            row[j] = pos[(int64_t)t * k + slot];
            wgt[j] = fni8::h2f(topw[(int64_t)t * k + slot]);
            ok[j] = row[j] >= 0 && row[j] < Tk;
        }
    }
    for (int h0 = threadIdx.x * 8; h0 < H; h0 += 256 * 8) {
        uint4 v[KM];
#pragma unroll
        for (int j = 0; j < KM; j++)
            v[j] = ok[j] ? *reinterpret_cast<const uint4*>(yr + row[j] * H + h0) : make_uint4(0, 0, 0, 0);
        uint16_t ob[8];
#pragma unroll
        for (int i = 0; i < 8; i++) ob[i] = 0;
#pragma unroll
        for (int j = 0; j < KM; j++) {
            if (!ok[j]) continue;
            const uint32_t w4[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint16_t c = (uint16_t)(w4[i >> 1] >> ((i & 1) * 16));
                const uint16_t pr = fni8::f2h(fni8::h2f(c) * wgt[j]);
                ob[i] = fni8::f2h(fni8::h2f(ob[i]) + fni8::h2f(pr));
            }
        }
        uint4 st;
        st.x = ob[0] | ((uint32_t)ob[1] << 16);
        st.y = ob[2] | ((uint32_t)ob[3] << 16);
        st.z = ob[4] | ((uint32_t)ob[5] << 16);
        st.w = ob[6] | ((uint32_t)ob[7] << 16);
        *reinterpret_cast<uint4*>(out + (int64_t)t * H + h0) = st;
    }
}

template <bool VEC>
__global__ __launch_bounds__(256) void moe_combine_kernel(
    const uint16_t* __restrict__ yr, int H, const int32_t* __restrict__ topi,
    const uint16_t* __restrict__ topw, const int32_t* __restrict__ pos, int k,
    int Tk, uint16_t* __restrict__ out) {
    const int t = blockIdx.x;
    int order[kMaxTopK];
    int eid[kMaxTopK];
    for (int j = 0; j < k; j++) {
        eid[j] = topi[(int64_t)t * k + j];
        order[j] = j;
    }
    for (int a = 1; a < k; a++) {  // insertion sort of the slots by expert id
        const int v = order[a];
        int b = a - 1;
        while (b >= 0 && eid[order[b]] > eid[v]) {
            order[b + 1] = order[b];
            b--;
        }
        order[b + 1] = v;
    }
    if constexpr (VEC) {
        for (int h0 = threadIdx.x * 8; h0 < H; h0 += 256 * 8) {
            float o[8];
            uint16_t ob[8];
#pragma unroll
            for (int i = 0; i < 8; i++) ob[i] = 0;
            for (int j = 0; j < k; j++) {
                const int slot = order[j];
                const float wgt = fni8::h2f(topw[(int64_t)t * k + slot]);
                const int64_t row = pos[(int64_t)t * k + slot];
                if (row < 0 || row >= Tk) continue;
                const uint4 v = *reinterpret_cast<const uint4*>(yr + row * H + h0);
                const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const uint16_t c = (uint16_t)(w4[i >> 1] >> ((i & 1) * 16));
                    const uint16_t pr = fni8::f2h(fni8::h2f(c) * wgt);
                    o[i] = fni8::h2f(ob[i]) + fni8::h2f(pr);
                    ob[i] = fni8::f2h(o[i]);
                }
            }
            uint4 st;
            st.x = ob[0] | ((uint32_t)ob[1] << 16);
            st.y = ob[2] | ((uint32_t)ob[3] << 16);
            st.z = ob[4] | ((uint32_t)ob[5] << 16);
            st.w = ob[6] | ((uint32_t)ob[7] << 16);
            *reinterpret_cast<uint4*>(out + (int64_t)t * H + h0) = st;
        }
    } else {
        for (int h = threadIdx.x; h < H; h += 256) {
            uint16_t ob = 0;
            for (int j = 0; j < k; j++) {
                const int slot = order[j];
                const float wgt = fni8::h2f(topw[(int64_t)t * k + slot]);
                const int64_t row = pos[(int64_t)t * k + slot];
                if (row < 0 || row >= Tk) continue;
                const uint16_t pr = fni8::f2h(fni8::h2f(yr[row * H + h]) * wgt);
                ob = fni8::f2h(fni8::h2f(ob) + fni8::h2f(pr));
            }
            out[(int64_t)t * H + h] = ob;
        }
    }
}

}  // namespace

namespace fni8h {

int launch_moe_sort(const int32_t* topi, int64_t T, int64_t k, int64_t E, int32_t* seg_off,
                    int32_t* row_token, int32_t* pos, hipStream_t st) {
    // us on MI355X by (ids, experts), 4 waves and 2 steps : 8 and 4 : 16 and 4 (and before,
    // walking 1024 ids at a time): (16, 128) 2.6 : 3.0 : 3.6 (3.3), (2048, 128) 3.3 :
    // 3.3 : 3.8 (6.0), (24000, 128) 18.8 : 11.3 : 8.3 (48.1).  More than one workgroup a
    // CU: (16, 512) 2.7 : 3.4 : 5.6 (3.4), (3000, 512) 4.0 : 4.1 : 6.0 (7.7), (24000, 512)
    // 16.5 : 10.9 : 11.5 (47.1).
#define FNI8_SORT(WAVES, KEEP)                                                                  \
    hipLaunchKernelGGL((moe_sort_kernel<WAVES, KEEP>), dim3((unsigned)E), dim3(WAVES * 64), 0, st, \
                       topi, (int)(T * k), (int)k, (int)E, seg_off, row_token, pos)
    if (T * k <= 2048) FNI8_SORT(4, 2);
    else if (E <= 256) FNI8_SORT(16, 4);
    else FNI8_SORT(8, 4);
#undef FNI8_SORT
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error_detail("moe_sort launch: %s", hipGetErrorString(e));
        return FNI8_ERR_LAUNCH;
    }
    return FNI8_OK;
}

int launch_moe_combine(const uint16_t* yr, int64_t H, const int32_t* topi,
                       const uint16_t* topw, const int32_t* pos, int64_t T, int64_t k,
                       uint16_t* out, hipStream_t st) {
    if (T == 0) return FNI8_OK;
    const bool vec = (H % 8 == 0) && ((uintptr_t)yr % 16 == 0) && ((uintptr_t)out % 16 == 0);
    if (vec && k <= 8)
        hipLaunchKernelGGL(moe_combine_small_kernel<8>, dim3((unsigned)T), dim3(256), 0, st, yr,
                           (int)H, topi, topw, pos, (int)k, (int)(T * k), out);
    else if (vec)
        hipLaunchKernelGGL(moe_combine_kernel<true>, dim3((unsigned)T), dim3(256), 0, st, yr,
                           (int)H, topi, topw, pos, (int)k, (int)(T * k), out);
    else
        hipLaunchKernelGGL(moe_combine_kernel<false>, dim3((unsigned)T), dim3(256), 0, st, yr,
                           (int)H, topi, topw, pos, (int)k, (int)(T * k), out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error_detail("moe_combine launch: %s", hipGetErrorString(e));
        return FNI8_ERR_LAUNCH;
    }
    return FNI8_OK;
}

}  // namespace fni8h
