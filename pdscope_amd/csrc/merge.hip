// K5: deterministic weighted merge back to token order, and the GPU half of
// the native CPU-group tail.
//   merge       restates the fused index_add_ merge of
//               expertbench/pdscope_runtime.py:450-469 as a gather: each
//               thread owns 8 output columns of one token and sums its k
//               rows in fp32, slot order, rounding once (no atomics).
//   merge_ordered restates the default per-expert merge of
//               pdscope_runtime.py:466-468 (merge='reference'): a token's k
//               rows are added in ascending expert id, each product rounded
//               to bf16 and each sum rounded to bf16, exactly as the
//               reference's sequence of per-expert bf16 index_add_ calls
//               (a token occurs once per expert, so each call is one add).
//               Grouped rows are sorted by expert, so ascending expert id is
//               ascending grouped row.
//   stage_merge restates native/native_layer_dispatch.cpp:83-88 (copy the
//               CPU block to device scratch, then index_add_ of
//               scratch * weights into out) in bf16 arithmetic, rows in order.
#include "common.h"

namespace pd {

// One output chunk of eight columns in either arithmetic.
template <bool ORDERED>
struct MergeAcc {
    float a[8];
    __device__ __forceinline__ void set(uint4 v) {
        a[0] = lo_bf(v.x); a[1] = hi_bf(v.x); a[2] = lo_bf(v.y); a[3] = hi_bf(v.y);
        a[4] = lo_bf(v.z); a[5] = hi_bf(v.z); a[6] = lo_bf(v.w); a[7] = hi_bf(v.w);
    }
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int q = 0; q < 8; ++q) a[q] = 0.0f;
    }
    // two columns: a = bf16(a + p)
    __device__ __forceinline__ void round_add(int q, float p0, float p1) {
        const uint32_t r = f2bf2_hw(a[q] + p0, a[q + 1] + p1);
        a[q] = lo_bf(r);
        a[q + 1] = hi_bf(r);
    }
    __device__ __forceinline__ void add(float w, uint4 v) {
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if constexpr (ORDERED) {
                const uint32_t p = f2bf2_hw(w * lo_bf(x[q]), w * hi_bf(x[q]));
                round_add(2 * q, lo_bf(p), hi_bf(p));
            } else {
                a[2 * q] = __builtin_fmaf(w, lo_bf(x[q]), a[2 * q]);
                a[2 * q + 1] = __builtin_fmaf(w, hi_bf(x[q]), a[2 * q + 1]);
            }
        }
    }
    __device__ __forceinline__ void add_last(uint4 v) {
        round_add(0, lo_bf(v.x), hi_bf(v.x));
        round_add(2, lo_bf(v.y), hi_bf(v.y));
        round_add(4, lo_bf(v.z), hi_bf(v.z));
        round_add(6, lo_bf(v.w), hi_bf(v.w));
    }
    __device__ __forceinline__ uint4 result() const {
        return make_uint4(f2bf2_hw(a[0], a[1]), f2bf2_hw(a[2], a[3]), f2bf2_hw(a[4], a[5]), f2bf2_hw(a[6], a[7]));
    }
};

// k <= KM: one wave per token and 64 output chunks (512 columns).  The
// token's k row indices and weights are the same for the whole wave: lane s
// holds slot s, the k values become scalars by lane reads, and up to eight rows
// of a lane's chunk are loaded before the first of them is added (sixteen leave
// room for fewer waves: T=1400, k=16, H=2048 18.9 us against 17.3, where one
// slot at a time took 17.4).
// Bound by the bytes of y.  ORDERED (rows in ascending grouped row, acc =
// bf16(acc + bf16(w * y)) per row, add_in added last): each lane ranks its
// slot against the others (k compares) and one lane push sorts them; a loop
// over all k for each next row in every thread took 71 us at T=4096, k=8,
// H=2048, 27 now (25 for the fp32 sum), and the roundings in integer
// arithmetic more than the loads (now the hardware's pair conversion).
template <int KM, bool ORDERED>
__global__ __launch_bounds__(256) void merge_kernel(const uint16_t *__restrict__ y,
                                                    const int32_t *__restrict__ row_of,
                                                    const uint16_t *__restrict__ w, int T, int k, int H,
                                                    const uint16_t *__restrict__ add_in,
                                                    uint16_t *__restrict__ out) {
    const int CH = H >> 3;
    const int groups = (CH + 63) >> 6;
    const int lane = lane_id();
    const int64_t total = (int64_t)T * groups;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int64_t item = (int64_t)blockIdx.x * 4 + wave; item < total; item += (int64_t)gridDim.x * 4) {
        const int t = (int)(item / groups), g = (int)(item - (int64_t)t * groups);
        const int c = g * 64 + lane;
        const bool live = c < CH;
        const int cc = live ? c : CH - 1;
        const size_t s0 = (size_t)t * k + min(lane, k - 1);
        int row = row_of[s0];
        int wb = w[s0];
        uint4 addv = make_uint4(0, 0, 0, 0);
        if (add_in) addv = reinterpret_cast<const uint4 *>(add_in + (size_t)t * H)[cc];
        if constexpr (ORDERED) {
            int rank = 0;
#pragma unroll
            for (int s = 0; s < KM; ++s)
                if (s < k) {
                    const int o = __builtin_amdgcn_readlane(row, s);
                    rank += (o < row) | ((o == row) & (s < lane));
                }
            // lane s's slot to lane `rank`; lanes past k keep to themselves
            const int dst = (lane < k ? rank : lane) * 4;
            row = __builtin_amdgcn_ds_permute(dst, row);
            wb = __builtin_amdgcn_ds_permute(dst, wb);
        }
        MergeAcc<ORDERED> acc;
        if (!ORDERED && add_in) acc.set(addv);
        else acc.zero();
#pragma unroll 1
        for (int b = 0; b < (KM > 8 ? k : 1); b += 8) {
            uint4 v[8];
#pragma unroll
            for (int s = 0; s < 8; ++s)
                if (b + s < k)
                    v[s] = reinterpret_cast<const uint4 *>(y + (size_t)__builtin_amdgcn_readlane(row, b + s) * H)[cc];
#pragma unroll
            for (int s = 0; s < 8; ++s)
                if (b + s < k) acc.add(bf2f((uint32_t)__builtin_amdgcn_readlane(wb, b + s)), v[s]);
        }
        if (ORDERED && add_in) acc.add_last(addv);
        if (live) reinterpret_cast<uint4 *>(out + (size_t)t * H)[c] = acc.result();
    }
}

// any k, one thread per chunk, one slot at a time
template <bool ORDERED>
__global__ __launch_bounds__(256) void merge_any_kernel(const uint16_t *__restrict__ y,
                                                        const int32_t *__restrict__ row_of,
                                                        const uint16_t *__restrict__ w, int T, int k, int H,
                                                        const uint16_t *__restrict__ add_in,
                                                        uint16_t *__restrict__ out) {
    const int CH = H >> 3;
    const int64_t total = (int64_t)T * CH;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int t = (int)(idx / CH), c = (int)(idx - (int64_t)t * CH);
        MergeAcc<ORDERED> acc;
        if (!ORDERED && add_in) acc.set(reinterpret_cast<const uint4 *>(add_in + (size_t)t * H)[c]);
        else acc.zero();
        if constexpr (ORDERED) {
            // the next larger grouped row each round
            int prev = -1;
            for (int n = 0; n < k; ++n) {
                int best = 0x7fffffff, bs = 0;
                for (int s = 0; s < k; ++s) {
                    const int r = row_of[(size_t)t * k + s];
                    if (r > prev && r < best) {
                        best = r;
                        bs = s;
                    }
                }
                prev = best;
                acc.add(bf2f(w[(size_t)t * k + bs]), reinterpret_cast<const uint4 *>(y + (size_t)best * H)[c]);
            }
        } else {
            for (int s = 0; s < k; ++s) {
                const int r = row_of[(size_t)t * k + s];
                acc.add(bf2f(w[(size_t)t * k + s]), reinterpret_cast<const uint4 *>(y + (size_t)r * H)[c]);
            }
        }
        if (ORDERED && add_in) acc.add_last(reinterpret_cast<const uint4 *>(add_in + (size_t)t * H)[c]);
        reinterpret_cast<uint4 *>(out + (size_t)t * H)[c] = acc.result();
    }
}

// rows whose token lies outside [0, out_rows) are skipped (never written)
__global__ __launch_bounds__(256) void stage_merge_kernel(const uint16_t *__restrict__ scratch, int64_t rows,
                                                          int H, const int64_t *__restrict__ tokens,
                                                          const uint16_t *__restrict__ weights, int64_t out_rows,
                                                          uint16_t *__restrict__ out) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= H) return;
    for (int64_t r = 0; r < rows; ++r) {
        const int64_t t = tokens[r];
        if (t < 0 || t >= out_rows) continue;
        const size_t o = (size_t)t * H + j;
        const float prod = bf16_round(bf2f(scratch[(size_t)r * H + j]) * bf2f(weights[r]));
        out[o] = (uint16_t)f2bf(bf2f(out[o]) + prod);
    }
}

}  // namespace pd

using namespace pd;

template <bool ORDERED>
static int launch_merge(const void *y, const int32_t *row_of, const void *w, int T, int k, int H,
                        const void *add_in, void *out, void *stream) {
    if (!y || !row_of || !w || !out) return fail(kEInval, "merge: null pointer");
    if (T < 1 || k < 1 || H < 8 || H % 8) return fail(kEInval, "merge: need T,k >= 1 and H % 8 == 0");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const uint16_t *yy = (const uint16_t *)y, *ww = (const uint16_t *)w, *aa = (const uint16_t *)add_in;
    if (k <= 16) {
        const int64_t waves = (int64_t)T * ((H / 8 + 63) / 64);
        const int blocks = (int)std::min<int64_t>((waves + 3) / 4, 65536);
        if (k <= 8)
            merge_kernel<8, ORDERED><<<blocks, 256, 0, s>>>(yy, row_of, ww, T, k, H, aa, (uint16_t *)out);
        else
            merge_kernel<16, ORDERED><<<blocks, 256, 0, s>>>(yy, row_of, ww, T, k, H, aa, (uint16_t *)out);
    } else {
        const int64_t total = (int64_t)T * (H / 8);
        const int blocks = (int)std::min<int64_t>((total + 255) / 256, 65536);
        merge_any_kernel<ORDERED><<<blocks, 256, 0, s>>>(yy, row_of, ww, T, k, H, aa, (uint16_t *)out);
    }
    return check_launch("merge_kernel");
}

PD_API int pdscope_merge(const void *y, const int32_t *row_of, const void *w, int T, int k, int H,
                         const void *add_in, void *out, void *stream) {
    return launch_merge<false>(y, row_of, w, T, k, H, add_in, out, stream);
}

PD_API int pdscope_merge_ordered(const void *y, const int32_t *row_of, const void *w, int T, int k, int H,
                                 const void *add_in, void *out, void *stream) {
    return launch_merge<true>(y, row_of, w, T, k, H, add_in, out, stream);
}

PD_API int pdscope_stage_merge(const void *host_block, int64_t rows, int64_t row_bytes, void *scratch,
                               void *out, const int64_t *tokens, const void *weights, int64_t out_rows,
                               void *stream) {
    if (!host_block || !scratch || !out || !tokens || !weights) return fail(kEInval, "stage_merge: null pointer");
    if (rows < 1 || row_bytes < 2 || row_bytes % 2) return fail(kEInval, "invalid decode pack shape");
    if (out_rows < 1) return fail(kEInval, "stage_merge: out needs at least one row");
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    hipError_t err = hipMemcpyAsync(scratch, host_block, (size_t)rows * (size_t)row_bytes, hipMemcpyHostToDevice, s);
    if (err != hipSuccess) return fail(kEHip, std::string("hipMemcpyAsync(stage): ") + hipGetErrorString(err));
    const int H = (int)(row_bytes / 2);
    stage_merge_kernel<<<(H + 255) / 256, 256, 0, s>>>((const uint16_t *)scratch, rows, H, tokens,
                                                       (const uint16_t *)weights, out_rows, (uint16_t *)out);
    return check_launch("stage_merge_kernel");
}
