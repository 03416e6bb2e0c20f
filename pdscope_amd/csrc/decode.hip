// K4: T == 1 decode expert FFN as a coalesced streaming GEMV, with the
// weighted merge fused into the down projection.
// Restates, for one token and its k routed experts, expert_forward
// (expertbench/adapters/qwen.py:87-90) as submitted per expert by the decode
// loop (expertbench/pdscope_runtime.py:326-350) and the merge
// (pdscope_runtime.py:450-469).
//
// Launch 1 (gate/up): one wave per two (expert, intermediate) items; every
//   lane streams 16-byte chunks of the gate and up rows (4 KiB rows at
//   H = 2048 are 4 chunks per lane), so each wave keeps 16 loads in flight.
//   h[s,i] = bf16(bf16(silu(bf16(g))) * bf16(u))  ->  h_ws [k, I]
// Launch 2 (down + merge): each 32-lane half-wave owns one expert row of
//   down_s (I bf16); a wave loads the rows of all k experts for its output
//   column j, two at a time per load, rounds each expert's y to bf16 (the expert
//   output dtype) and
//   accumulates w_s * y_s in fp32 in slot order (merge_mode 0:
//   out[j] = bf16(sum_s w_s * y_s[j]), one rounding), or keeps the y_s and
//   adds them in ascending expert id in bf16 arithmetic (merge_mode 1, the
//   reference's merge, expertbench/pdscope_runtime.py:466-468:
//   acc = bf16(acc + bf16(w_s * y_s[j]))).  h (k*I bf16) is staged in LDS
//   once per block.  Always-on shared experts are a further row per output
//   column; their gate/up half runs beside the router (route.hip).
#include "common.h"
#include "topk.h"

namespace pd {

template <int NJ>
__global__ __launch_bounds__(256) void decode_gateup_kernel(const uint16_t *__restrict__ x,
                                                            const int32_t *__restrict__ ids,
                                                            const uint16_t *const *__restrict__ slots, int H,
                                                            int I, int k, uint16_t *__restrict__ h_ws) {
    const int lane = lane_id();
    const int q0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 2;
    const int items = k * I;
    if (q0 >= items) return;
    // lane owns 16-byte chunks lane + 64*j (j < NJ) of each H-row; when H is
    // not a multiple of 512 the tail chunks are clamped and masked out
    const int C = H >> 3;
    uint4 xv[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) xv[j] = reinterpret_cast<const uint4 *>(x)[min(lane + 64 * j, C - 1)];
    uint4 gv[2][NJ], uv[2][NJ];
    bool ok[2];
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const int q = min(q0 + it, items - 1);
        const int s = q / I, i = q - s * I;
        const uint16_t *base = slots[ids[s]];
        // an expert without a ready copy reads the activation row instead
        // (H elements, in bounds) and contributes h = 0
        ok[it] = base != nullptr;
        const uint4 *grow = ok[it] ? reinterpret_cast<const uint4 *>(base + (size_t)i * H)
                                   : reinterpret_cast<const uint4 *>(x);
        const uint4 *urow = ok[it] ? reinterpret_cast<const uint4 *>(base + (size_t)(I + i) * H)
                                   : reinterpret_cast<const uint4 *>(x);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            gv[it][j] = ld_nt(grow + min(lane + 64 * j, C - 1));
            uv[it][j] = ld_nt(urow + min(lane + 64 * j, C - 1));
        }
    }
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        float g = 0.0f, u = 0.0f;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            if (lane + 64 * j < C) {
                g = dot8(gv[it][j], xv[j], g);
                u = dot8(uv[it][j], xv[j], u);
            }
        }
        g = wave_sum_dpp(g);
        u = wave_sum_dpp(u);
        const int q = q0 + it;
        if (lane == 0 && q < items) {
            const float a = bf16_round(silu_f32(bf16_round(g)));
            h_ws[q] = ok[it] ? (uint16_t)f2bf(a * bf16_round(u)) : (uint16_t)0;
        }
    }
}

// Down half of always-on shared experts in the same launch (slot == nullptr: none).
struct SharedDown {
    const uint16_t *const *slot;  // [1] gate|up|down block
    int I;
    const uint16_t *h;            // [I]
    uint16_t *y;                  // [H]
};

// CPL = 16-byte chunks per lane per expert row (ceil(I / 8 / 32)); KP slot
// pairs (k <= 2 KP) and CS 16-byte chunks per lane of a shared row (0: none).
// Every row of the wave's output column is loaded before h is staged, so the
// launch, bound by the bytes of the down rows, pays one memory latency instead
// of one per slot pair (two waves a SIMD cannot hide it).  A pair that an odd k
// leaves half empty reads its other half's row twice, in the same loads; with
// h read there instead (and k <= 2 on two pairs) both decode launches took
// 9.4 us against 7.7 at k = 1, 10.3 against 8.7 at k = 2 and 18.2 against 16.9
// at k = 7 (H 2048, I 768; one slot pair at a time 8.1, 9.1 and 20.5).
template <int CPL, int KP, int CS>
__global__ __launch_bounds__(256) void decode_down_kernel(const uint16_t *__restrict__ h_ws,
                                                          const int32_t *__restrict__ ids,
                                                          const uint16_t *__restrict__ w,
                                                          const uint16_t *const *__restrict__ slots, int H,
                                                          int I, int k, int merge_mode, SharedDown sd,
                                                          uint16_t *__restrict__ out) {
    extern __shared__ uint4 s_h[];         // k * I, then sd.I bf16
    __shared__ float s_ys[4][2 * KP];      // per wave: bf16 y of each slot
    const int CI = I >> 3, CSI = CS ? sd.I >> 3 : 0;
    const int lane = lane_id(), half = lane >> 5, hl = lane & 31, wave = threadIdx.x >> 6;
    const int j = blockIdx.x * 4 + wave;
    const int jc = min(j, H - 1);
    const size_t IH2 = 2 * (size_t)I * H;
    uint4 wv[KP][CPL];
    bool has[KP];
#pragma unroll
    for (int p = 0; p < KP; ++p) {
        // past the last slot: the last slot's row again, which the other half reads
        const uint16_t *base = slots[ids[min(2 * p + half, k - 1)]];
        has[p] = base != nullptr;
        // no ready copy: read h itself (k*I elements, in bounds) and add 0
        const uint4 *row = base ? reinterpret_cast<const uint4 *>(base + IH2 + (size_t)jc * I)
                                : reinterpret_cast<const uint4 *>(h_ws);
#pragma unroll
        for (int c = 0; c < CPL; ++c) wv[p][c] = ld_nt(row + min(hl + 32 * c, CI - 1));
    }
    // lane s: slot s's expert id and weight, in ascending expert id for merge_mode 1
    int order = lane, wb = 0;
    if (lane < k) wb = w[lane];
    if (merge_mode) {
        const int e = lane < k ? ids[lane] : 0;
        int rank = 0;
        for (int s = 0; s < k; ++s) rank += __builtin_amdgcn_readlane(e, s) < e;
        const int dst = (lane < k ? rank : lane) * 4;
        order = __builtin_amdgcn_ds_permute(dst, lane);
        wb = __builtin_amdgcn_ds_permute(dst, wb);
    }
    uint4 sv[CS ? CS : 1];
    bool shas = false;
    if constexpr (CS > 0) {
        const uint16_t *base = sd.slot[0];
        shas = base != nullptr;
        const uint4 *row = base ? reinterpret_cast<const uint4 *>(base + 2 * (size_t)sd.I * H + (size_t)jc * sd.I)
                                : reinterpret_cast<const uint4 *>(sd.h);
#pragma unroll
        for (int c = 0; c < CS; ++c) sv[c] = ld_nt(row + min(lane + 64 * c, CSI - 1));
    }
    for (int idx = threadIdx.x; idx < k * CI; idx += blockDim.x)
        s_h[idx] = reinterpret_cast<const uint4 *>(h_ws)[idx];
    for (int idx = threadIdx.x; idx < CSI; idx += blockDim.x)
        s_h[k * CI + idx] = reinterpret_cast<const uint4 *>(sd.h)[idx];
    __syncthreads();
#pragma unroll
    for (int p = 0; p < KP; ++p) {
        const int s = min(2 * p + half, k - 1);
        float acc = 0.0f;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            const int ch = hl + 32 * c;
            if (ch < CI) acc = dot8(wv[p][c], s_h[s * CI + ch], acc);
        }
        acc = half_sum_dpp(has[p] ? acc : 0.0f);  // lanes 31 / 63 hold the sums of the two halves
        if (hl == 31 && 2 * p + half < k) s_ys[wave][2 * p + half] = bf16_round(acc);
    }
    float add = 0.0f;
    if constexpr (CS > 0) {
        float acc = 0.0f;
#pragma unroll
        for (int c = 0; c < CS; ++c) {
            const int ch = lane + 64 * c;
            if (ch < CSI) acc = dot8(sv[c], s_h[k * CI + ch], acc);
        }
        add = bf16_round(wave_sum_dpp(shas ? acc : 0.0f));
    }
    wave_lds_sync();
    // the weighted sum in either merge arithmetic; the shared experts' y is
    // unweighted: first in the fp32 sum, last in the bf16 sequence
    float total = merge_mode ? 0.0f : add;
    for (int s = 0; s < k; ++s) {
        const float ws = bf2f((uint32_t)__builtin_amdgcn_readlane(wb, s));
        const float ys = s_ys[wave][__builtin_amdgcn_readlane(order, s)];
        total = merge_mode ? bf16_round(total + bf16_round(ws * ys)) : __builtin_fmaf(ws, ys, total);
    }
    if (CS > 0 && merge_mode) total = bf16_round(total + add);
    if (lane == 0 && j < H) {
        if constexpr (CS > 0) sd.y[j] = (uint16_t)f2bf(add);
        out[j] = (uint16_t)f2bf(total);
    }
}

// any shape the entry point takes: one slot pair at a time
template <int CPL>
__global__ __launch_bounds__(256) void decode_down_any_kernel(const uint16_t *__restrict__ h_ws,
                                                              const int32_t *__restrict__ ids,
                                                              const uint16_t *__restrict__ w,
                                                              const uint16_t *const *__restrict__ slots, int H,
                                                              int I, int k, int merge_mode,
                                                              uint16_t *__restrict__ out) {
    extern __shared__ uint4 s_h[];
    __shared__ float s_ys[4][16];  // per wave: bf16 y of each slot
    const int CI = I >> 3;
    for (int idx = threadIdx.x; idx < k * CI; idx += blockDim.x)
        s_h[idx] = reinterpret_cast<const uint4 *>(h_ws)[idx];
    __syncthreads();
    const int lane = lane_id(), half = lane >> 5, hl = lane & 31;
    const int j = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (j >= H) return;
    const size_t IH2 = 2 * (size_t)I * H;
    float total = 0.0f;
    for (int p = 0; p < k; p += 2) {
        const int s = p + half;
        float acc = 0.0f;
        if (s < k) {
            const uint16_t *base = slots[ids[s]];
            // no ready copy: read h itself (k*I elements, in bounds) and add 0
            const uint4 *row = base ? reinterpret_cast<const uint4 *>(base + IH2 + (size_t)j * I)
                                    : reinterpret_cast<const uint4 *>(h_ws);
            uint4 wv[CPL];
#pragma unroll
            for (int c = 0; c < CPL; ++c) wv[c] = ld_nt(row + min(hl + 32 * c, CI - 1));
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                const int ch = hl + 32 * c;
                if (ch < CI) acc = dot8(wv[c], s_h[s * CI + ch], acc);
            }
            if (!base) acc = 0.0f;
        }
        acc = half_sum_dpp(acc);  // lanes 31 / 63 hold the sums of the two halves
        const float even = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(acc), 31));
        const float odd = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(acc), 63));
        if (lane == 0) {
            total = __builtin_fmaf(bf2f(w[p]), bf16_round(even), total);
            if (p + 1 < k) total = __builtin_fmaf(bf2f(w[p + 1]), bf16_round(odd), total);
            s_ys[threadIdx.x >> 6][p] = bf16_round(even);
            if (p + 1 < k) s_ys[threadIdx.x >> 6][p + 1] = bf16_round(odd);
        }
    }
    if (lane == 0 && merge_mode) {
        const float *ys = s_ys[threadIdx.x >> 6];
        total = 0.0f;
        int prev = -1;
        for (int n = 0; n < k; ++n) {  // the next larger expert id each round
            int best = 0x7fffffff, bs = 0;
            for (int s = 0; s < k; ++s) {
                const int e = ids[s];
                if (e > prev && e < best) {
                    best = e;
                    bs = s;
                }
            }
            prev = best;
            total = bf16_round(total + bf16_round(bf2f(w[bs]) * ys[bs]));
        }
    }
    if (lane == 0) out[j] = (uint16_t)f2bf(total);
}

}  // namespace pd

using namespace pd;

// Slot pairs, chunks per half-wave lane and shared chunks per lane that
// decode_down_kernel is built for; false: decode_down_any_kernel (no shared).
static bool down_fits(int k, int I, int shared_I) {
    return k <= 8 && I <= 6 * 256 && shared_I <= 6 * 512;
}

static int launch_decode(const void *x, const int32_t *ids, const void *w, int k, const void *const *slots, int H,
                         int I, void *h_ws, void *out, int merge_mode, SharedDown sd, void *stream) {
    if (!x || !ids || !w || !slots || !h_ws || !out) return fail(kEInval, "decode: null pointer");
    if (merge_mode != 0 && merge_mode != 1) return fail(kEInval, "decode: merge_mode must be 0 or 1");
    if (k < 1 || k > 16) return fail(kEInval, "decode: need 1 <= k <= 16");
    if (H < 8 || H % 8 || H > 4096) return fail(kEInval, "decode: need H % 8 == 0 and H <= 4096");
    if (I < 8 || I % 8 || I > 8192) return fail(kEInval, "decode: need I % 8 == 0 and I <= 8192");
    if (((size_t)k * I + sd.I) * 2 > 64 * 1024) return fail(kEInval, "decode: k*I*2 must fit 64 KiB of LDS");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const uint16_t *xp = (const uint16_t *)x;
    const uint16_t *const *sp = (const uint16_t *const *)slots;
    const int waves = (k * I + 1) / 2;
    const int blocks = (waves + 3) / 4;
    switch ((H / 8 + 63) / 64) {
#define PD_GU(NJ)                                                                                          \
    case NJ:                                                                                               \
        decode_gateup_kernel<NJ><<<blocks, 256, 0, s>>>(xp, ids, sp, H, I, k, (uint16_t *)h_ws);           \
        break;
        PD_GU(1) PD_GU(2) PD_GU(3) PD_GU(4) PD_GU(5) PD_GU(6) PD_GU(7) PD_GU(8)
#undef PD_GU
    default:
        return fail(kEInval, "decode: unsupported H");
    }
    int rc = check_launch("decode_gateup_kernel");
    if (rc) return rc;
    const int cpl = ((I >> 3) + 31) / 32;
    const size_t lds = ((size_t)k * I + sd.I) * 2;
    const int dblocks = (H + 3) / 4;
    const uint16_t *hp = (const uint16_t *)h_ws, *wp = (const uint16_t *)w;
    if (down_fits(k, I, sd.I)) {
        const int kp = k <= 2 ? 1 : k <= 4 ? 2 : k <= 6 ? 3 : 4, cs = sd.slot ? (sd.I <= 3 * 512 ? 3 : 6) : 0;
        const int cc = cpl <= 3 ? 3 : 6;
#define PD_DN(C, P, S)                                                                                          \
    if (cc == C && kp == P && cs == S)                                                                          \
        decode_down_kernel<C, P, S><<<dblocks, 256, lds, s>>>(hp, ids, wp, sp, H, I, k, merge_mode, sd, (uint16_t *)out);
#define PD_DNS(C, P) PD_DN(C, P, 0) PD_DN(C, P, 3) PD_DN(C, P, 6)
        PD_DNS(3, 1) PD_DNS(3, 2) PD_DNS(3, 3) PD_DNS(3, 4) PD_DNS(6, 1) PD_DNS(6, 2) PD_DNS(6, 3) PD_DNS(6, 4)
#undef PD_DNS
#undef PD_DN
        return check_launch("decode_down_kernel");
    }
    if (sd.slot) return fail(kEInval, "decode: shared experts need k <= 8, I <= 1536 and a shared I <= 3072");
    switch (cpl) {
#define PD_DN(C)                                                                                           \
    case C:                                                                                                \
        decode_down_any_kernel<C><<<dblocks, 256, lds, s>>>(hp, ids, wp, sp, H, I, k, merge_mode, (uint16_t *)out); \
        break;
        PD_DN(1) PD_DN(2) PD_DN(3) PD_DN(4) PD_DN(5) PD_DN(6) PD_DN(7) PD_DN(8)
#undef PD_DN
    default:
        if (cpl <= 32) {
            decode_down_any_kernel<32><<<dblocks, 256, lds, s>>>(hp, ids, wp, sp, H, I, k, merge_mode,
                                                                 (uint16_t *)out);
        } else {
            return fail(kEInval, "decode: unsupported I");
        }
    }
    return check_launch("decode_down_kernel");
}

PD_API int pdscope_swiglu_decode(const void *x, const int32_t *ids, const void *w, int k,
                                 const void *const *slots, int H, int I, void *h_ws, void *out,
                                 int merge_mode, void *stream) {
    return launch_decode(x, ids, w, k, slots, H, I, h_ws, out, merge_mode, SharedDown{nullptr, 0, nullptr, nullptr},
                         stream);
}

PD_API int pdscope_swiglu_decode_shared(const void *x, const int32_t *ids, const void *w, int k,
                                        const void *const *slots, int H, int I, void *h_ws,
                                        const void *const *shared_slot, int shared_I, const void *h_shared,
                                        void *y_shared, void *out, int merge_mode, void *stream) {
    if (!shared_slot || !h_shared || !y_shared || shared_I < 8 || shared_I % 8)
        return fail(kEInval, "decode_shared: bad shared arguments");
    return launch_decode(x, ids, w, k, slots, H, I, h_ws, out, merge_mode,
                         SharedDown{(const uint16_t *const *)shared_slot, shared_I, (const uint16_t *)h_shared,
                                    (uint16_t *)y_shared},
                         stream);
}

// Whether pdscope_route_topk_shared + pdscope_swiglu_decode_shared run one
// token of this shape.
PD_API int pdscope_decode_shared_supported(int H, int I, int E, int k, int shared_I) {
    return H >= 16 && H % 16 == 0 && H <= 4096 && I >= 8 && I % 8 == 0 && E >= 32 && E <= 256 && E % 32 == 0 &&
           k >= 1 && k <= E && shared_I >= 8 && shared_I % 8 == 0 && down_fits(k, I, shared_I) &&
           ((size_t)k * I + shared_I) * 2 <= 64 * 1024;
}
