// K3: grouped SwiGLU expert FFN for prefill on bf16 MFMA (gfx950).
// Restates expert_forward (expertbench/adapters/qwen.py:87-90) for every
// selected expert at once, replacing the per-expert launches of
// ExpertExecutor.gpu (expertbench/executor.py:454-488).
//
// Two launches per call:
//   gate/up : h[r,i] = bf16(bf16(silu(bf16(x_r.gate_i))) * bf16(x_r.up_i))
//             the A rows are gathered through perm_token, the B tile holds
//             BN/2 gate rows and the matching BN/2 up rows, so the SwiGLU
//             epilogue pairs accumulators of the same lane;
//   down    : y[r,n] = bf16(h_r . down_n)
// Both operands are K-contiguous ([rows, K] activations, [out, in] weights),
// so every 16-byte chunk feeds one MFMA lane directly.  Tiles stream into
// multi-stage LDS rings by direct-to-LDS loads (global_load_lds_dwordx4)
// with a 16-byte-chunk XOR swizzle applied on the source side (see Geo),
// so fragment reads are bank-conflict free.
// MFMA: v_mfma_f32_32x32x16_bf16, fp32 accumulation.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace pd {

// LDS tile geometry for a K step of BK bf16 elements: a tile row is BK * 2
// bytes (CPR chunks of 16 B); one wave-wide direct-to-LDS load fills 1 KB,
// i.e. RPI consecutive rows.  With 64 banks of 4 bytes, a 16-byte fragment
// read serves 16 lanes (16 consecutive rows, one logical chunk) per cycle;
// rows share a 256-byte bank line in groups of RPL, so chunk c of row r is
// stored in slot c ^ ((r / RPL) % CPR) and the 16 rows of a fragment read
// land in 16 distinct 16-byte bank groups (conflict free).
template <int BK>
struct Geo {
    static constexpr int RB = BK * 2;
    static constexpr int CPR = BK / 8;
    static constexpr int RPI = 1024 / RB;
    static constexpr int RPL = 256 / RB;
    static __device__ __forceinline__ int key(int r) { return (r / RPL) % CPR; }
    static __device__ __forceinline__ int off(int r, int c) { return r * RB + ((c ^ key(r)) << 4); }
};

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(1))) const void g_void_t;

// One wave-wide direct-to-LDS load: lane l's 16 bytes at src land at
// dst + 16 l (dst is wave-uniform), bypassing the registers.  AUX is the
// cache-policy field.  kDeviceScope (sc1) makes the load device-coherent, so
// it is served by the L2 without allocating in the CU's vector L1; kStream
// (nt) marks the lines as not to be kept.  A weight tile is read once per
// m-tile of its expert: where the expert has one m-tile nothing will ask for
// it again, and streaming reads run at 7.0 TB/s against 6.3 and leave the L2
// to the activations; where it has more, the m-tiles read it at about the
// same time and the second should hit the L2.  Chosen per tile, against sc1
// throughout: Qwen shape T=201 gate/up 143 -> 128 us, down 79 -> 71; T=512
// 145 -> 135 and 83 -> 76; T=4096 (about half the experts have two tiles)
// 289 -> 284 and 167 -> 160; DeepSeek-V2-Lite shape T=1304 down 95 -> 82.
// nt throughout: T=512 with Zipf routing 159 against 148, T=4096 301.
// Streamed lines are not kept in the Infinity Cache either, so a pass whose
// weights all fit there (256 MB) and that is repeated at once is the one that
// loses: 16 experts of the Qwen shape, gate/up again and again, 19.8 us under
// sc1 and 28.8 here (32.3 and 29.3 when other experts come in between; weights
// just copied from the host 34.3 and 29.7, 4 experts); one layer of T=2 57.0
// and 59.5, two layers in turn 65.0 and 57.3.
// Activation tiles keep the default policy.
constexpr int kDeviceScope = 16;
constexpr int kStream = 2;
template <int AUX = 0>
__device__ __forceinline__ void load_lds16(const uint16_t *src, uint8_t *dst) {
    __builtin_amdgcn_global_load_lds((g_void_t *)(uintptr_t)src, (lds_void_t *)(uint32_t)(uintptr_t)dst, 16, 0, AUX);
}

// Hides a per-lane load offset from loop-invariant code motion, so each
// 64-bit address (uniform base + offset) is formed next to its load instead
// of being hoisted out of the K loop as a live register pair per load.
__device__ __forceinline__ void opaque(uint32_t &v) { asm volatile("" : "+v"(v)); }

// Wait until at most n vector-memory operations of this wave are in flight
// (n is a compile-time constant in every use).
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// wait_vm<n> for a wave-uniform n in [0, 24] known only at run time
__device__ __forceinline__ void wait_vm_rt(int n) {
#define PD_W(K) else if (n == K) wait_vm<K>();
    if (n <= 0) wait_vm<0>();
    PD_W(1) PD_W(2) PD_W(3) PD_W(4) PD_W(5) PD_W(6) PD_W(7) PD_W(8) PD_W(9) PD_W(10) PD_W(11) PD_W(12)
    PD_W(13) PD_W(14) PD_W(15) PD_W(16) PD_W(17) PD_W(18) PD_W(19) PD_W(20) PD_W(21) PD_W(22) PD_W(23)
    else wait_vm<24>();
#undef PD_W
}

// Workgroup barrier for the LDS ring.  __syncthreads() would also wait for
// every outstanding direct-to-LDS load (its release fence covers them) and
// drain the pipeline; here the caller waits for exactly the stage it needs
// (wait_stage), this wave's LDS reads are complete (lgkmcnt 0) before the
// slot they read can be refilled, and the memory clobber keeps the
// compiler from moving LDS accesses across the barrier.
__device__ __forceinline__ void ring_barrier() {
    // lgkmcnt(0) through the builtin, so the compiler's own wait analysis
    // knows every earlier LDS read has completed here
    __builtin_amdgcn_s_waitcnt(0xc07f);
    asm volatile("s_barrier" ::: "memory");
}

// Wait until the stage to be consumed has landed, `younger` (0 .. S-2)
// later stages of LPW loads each being allowed to stay in flight.
template <int S, int LPW, int Y = S - 2>
__device__ __forceinline__ void wait_stage(int younger) {
    if constexpr (Y <= 0) {
        wait_vm<0>();
    } else {
        if (younger >= Y) {
            wait_vm<Y * LPW>();
            return;
        }
        wait_stage<S, LPW, Y - 1>(younger);
    }
}

// Always-on shared experts as further tiles of a grouped launch (slot ==
// nullptr: none): one MLP of intermediate I over rows 0 .. T-1 in order, on the
// launch's own tile shape.  Its tiles take the first blocks of the grid: the
// down half is the longest tile of the launch (K = shared I).  As launches of
// their own on a second stream, on 256-row tiles that read the shared block
// fewest times, they held CUs for long while the routed launches waited at the
// join (48 blocks for the down half at T=1304), and their time moved with how
// the two streams met.  DeepSeek-V2-Lite layer, then and now (today's loads and
// stores among it): T=48 233 -> 199 us, T=128 243 -> 222, T=180 248 -> 228 (six
// 32-row tiles), T=190 244 -> 239, T=400 257 -> 256 and T=470 272 -> 260 (eight
// 64-row tiles), T=640 272 -> 257, T=1304 324 -> 307, T=2048 390 -> 392, T=4096
// 699 -> 697.
struct SharedTiles {
    const uint16_t *const *slot;  // [1] gate|up|down block
    int I, T;
    uint16_t *h;                  // [T, I]
    uint16_t *y;                  // [T, H]
};

template <int BM, int BN, int BK, int SA, int SB>
constexpr int kRingBytes = (SA * BM + SB * BN) * BK * 2;

// Tile BM x BN x BK, WM x WN waves (4 or 8: with 8, two waves share each
// SIMD so one wave's MFMAs cover the other's LDS reads, waits and
// epilogue).  OCC is the number of workgroups per CU the tile is sized for
// (LDS and registers): with 2, one workgroup's ring fill and epilogue
// overlap the other's K loop.  The A tile (activation rows) and the B tile (weight rows)
// stream into two LDS rings of SA and SB stages by direct-to-LDS loads.
// With SA == SB every wave loads its share of both.  With SA != SB
// (8 waves) the first half of the waves loads only A and the second half
// only B: a wave's load counter completes in issue order, so a wave that
// loads both operands cannot keep the slow weight stream (HBM) further
// ahead than the fast activation gathers (L2 / Infinity Cache); split
// roles let the B ring run SB-1 stages ahead on its own.  Every wave
// computes.  ILV deals the tile's 32-row blocks to the WM wave rows
// round-robin (block b to wave row b % WM) instead of in contiguous runs, so
// a tile whose experts fill only part of its rows keeps the MFMA work of
// every SIMD about equal.  Tiles are numbered (m-tile, n-tile) with n fastest and the
// tile range is cut into 8 contiguous pieces, one per XCD (block b runs on
// XCD b % 8): all n-tiles of an m-tile share the gathered activation rows
// in one L2, and the m-tiles of one expert read the same weight tiles at
// the same time from one L2.
template <int BM, int BN, int BK, int WM, int WN, int SA, int SB, bool ILV, bool GATEUP, int OCC, int FK>
__device__ __forceinline__ void grouped_tile(
    uint8_t *smem, const uint16_t *__restrict__ a_src, const int32_t *__restrict__ perm_token,
    const int32_t *__restrict__ offsets, const int32_t *__restrict__ sel, int nsel,
    const int32_t *__restrict__ tile_start, const uint16_t *const *__restrict__ slots, int H, int I_routed,
    uint16_t *__restrict__ out_routed, const SharedTiles &sh) {
    constexpr int NW = WM * WN;
    static_assert(NW == 4 || NW == 8, "4 or 8 waves");
    constexpr bool SPLIT = SA != SB;
    static_assert(!SPLIT || NW == 8, "split load roles need 8 waves");
    constexpr int TM = BM / WM, TN = BN / WN;  // wave tile
    constexpr int MB = TM / 32, NB = TN / 32;  // 32x32 MFMA blocks per wave
    static_assert(MB >= 1 && NB >= 1 && (!GATEUP || NB % 2 == 0), "wave tiling");
    static_assert(MB <= 4, "the live row-block dispatch below covers up to 4 row blocks per wave");
    typedef Geo<BK> G;
    constexpr int NWA = SPLIT ? NW / 2 : NW, NWB = SPLIT ? NW / 2 : NW;  // waves loading A / B
    constexpr int AL = BM / G::RPI / NWA, BL = BN / G::RPI / NWB;  // 1 KB loads per loading wave per stage
    static_assert(AL >= 1 && BL >= 1 && AL * G::RPI * NWA == BM && BL * G::RPI * NWB == BN, "tile / load shape");
    static_assert(!SPLIT || (SA - 1) * AL <= 24, "A-wave waits count live loads up to wait_vm_rt's range");
    constexpr int ASTAGE = BM * G::RB, BSTAGE = BN * G::RB;
    static_assert(OCC * (SA * ASTAGE + SB * BSTAGE) <= 160 * 1024, "LDS of OCC workgroups per CU");
    static_assert(SA * ASTAGE + SB * BSTAGE == kRingBytes<BM, BN, BK, SA, SB>, "LDS ring");
    uint8_t *const ring_a = smem;
    uint8_t *const ring_b = smem + SA * ASTAGE;

    // ---- tile -> (m-tile, n-tile): the shared tiles' blocks, then the routed ones'
    const int nts = GATEUP ? sh.I / (BN / 2) : H / BN;
    const int stotal = sh.slot ? (sh.T + BM - 1) / BM * nts : 0;
    const int sblocks = (stotal + 7) & ~7;
    const bool shared = (int)blockIdx.x < sblocks;
    const int I = shared ? sh.I : I_routed;
    const int NT = GATEUP ? I / (BN / 2) : H / BN;
    const int total = shared ? stotal : tile_start[nsel] * NT;
    const int bid = shared ? blockIdx.x : blockIdx.x - sblocks;
    const int per_xcd = (total + 7) >> 3;
    const int pos = bid >> 3;
    if (pos >= per_xcd) return;
    const int t = (bid & 7) * per_xcd + pos;
    if (t >= total) return;
    const int mt = t / NT, nt = t - mt * NT;
    int row0 = 0, row_end = sh.T, m0 = mt * BM;  // the expert's rows, the tile's first row
    const uint16_t *base;
    if (shared) {
        base = sh.slot[0];
    } else {
        // the expert position of m-tile mt: the last lo with tile_start[lo] <= mt.
        // tile_start is non-decreasing with tile_start[0] = 0, so lo is the count
        // of j in [1, nsel) with tile_start[j] <= mt: independent loads and a
        // ballot per 64 entries instead of a chain of dependent loads
        int lo = 0;
#pragma unroll 4
        for (int b0 = 1; b0 < nsel; b0 += 64) {
            const int j = b0 + (threadIdx.x & 63);
            lo += __popcll(__ballot(j < nsel && tile_start[j] <= mt));
        }
        lo = __builtin_amdgcn_readfirstlane(lo);
        const int e = sel[lo];
        row0 = offsets[e];
        row_end = offsets[e + 1];
        m0 = row0 + (mt - tile_start[lo]) * BM;
        base = slots[e];
    }
    const int K = GATEUP ? H : I;
    const int n0 = nt * (GATEUP ? BN / 2 : BN);  // first intermediate (gate/up) or output column
    uint16_t *const out = shared ? (GATEUP ? sh.h : sh.y) : out_routed;
    if (base == nullptr) {
        // no ready copy: never dereferenced.  Routed rows keep what y holds
        // (another launch may have written them); y of the shared experts is
        // added to every token, so without a copy it is zero
        if (shared && !GATEUP)
            for (int c = threadIdx.x; c < min(BM, row_end - m0) * (BN / 8); c += 64 * NW)
                st_through(out + (size_t)(m0 + c / (BN / 8)) * H + n0 + c % (BN / 8) * 8, make_uint4(0, 0, 0, 0));
        return;
    }
    const size_t IH = (size_t)I * H;

    // ---- per-lane source rows: load q of A-wave wa covers A rows
    // RPI(wa + NWA q) .. +RPI-1 (B likewise with wb, NWB); lane l takes row
    // +l/CPR and the logical chunk that belongs in slot l % CPR of that row
    // (the swizzle).
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool a_role = !SPLIT || wave < NWA;
    const int wa = wave, wb = SPLIT ? wave - NWA : wave;
    const int rl = lane / G::CPR, slot = lane % G::CPR;
    // A loads whose rows all lie past the expert's last row are not issued (split roles only: there an A wave's load count per stage
    // is its own, and its waits count its live loads); their LDS rows keep
    // stale values, which reach only accumulator rows the epilogue skips
    const int live_groups = (min(row_end - m0, BM) + G::RPI - 1) / G::RPI;
    const int a_live = SPLIT ? __builtin_amdgcn_readfirstlane(
                                   min(AL, max(0, (live_groups - wa + NWA - 1) / NWA)))
                             : AL;
    // Load addresses.  Load q of a wave covers rows (w + NW q) RPI .. + RPI-1 of
    // its tile, and NW RPI is a multiple of the swizzle period (16 rows), so
    // a lane's row within the group and its swizzled chunk are the same for
    // every q: a per-lane byte offset plus a wave-uniform part per q.  Only the
    // gathered gate/up activation rows need a register per load (their token
    // offsets, in 16-byte units from a_src: 2^32 units cover 64 GiB).
    static_assert((NWA * G::RPI) % 16 == 0 && (NWB * G::RPI) % 16 == 0, "swizzle period");
    const uint32_t a_cs = (uint32_t)(slot ^ G::key(wa * G::RPI + rl));
    const uint32_t b_cs = (uint32_t)(slot ^ G::key(wb * G::RPI + rl));
    uint32_t lp[GATEUP ? AL : 1];
    if (GATEUP && a_role) {
#pragma unroll
        for (int q = 0; q < AL; ++q) {
            const int gr = min(m0 + (wa + NWA * q) * G::RPI + rl, row_end - 1);
            lp[q] = (uint32_t)(shared ? gr : perm_token[gr]) * (uint32_t)(H / 8) + a_cs;
        }
    }
    // B: the lane's row and chunk in bytes from the first row of its load group
    const uint32_t b_lane = (uint32_t)rl * (uint32_t)(K * 2) + b_cs * 16u;
    // B: byte offset of load q's first row in the expert's block
    auto b_row0 = [&](int q) __attribute__((always_inline)) {
        const int rb = (wb + NWB * q) * G::RPI;
        if (GATEUP)
            return rb < BN / 2 ? (size_t)(n0 + rb) * H * 2 : (size_t)IH * 2 + (size_t)(n0 + rb - BN / 2) * H * 2;
        return (size_t)IH * 4 + (size_t)(n0 + rb) * I * 2;
    };
    const uint8_t *const a_base = reinterpret_cast<const uint8_t *>(shared && !GATEUP ? sh.h : a_src);
    const uint8_t *const b_base = reinterpret_cast<const uint8_t *>(base);
    const bool one_tile = row_end - row0 <= BM;  // no other m-tile reads these weights
    const int KT = K / BK;
    auto issue_a = [&](int kt) __attribute__((always_inline)) {
        uint8_t *st = ring_a + (kt % SA) * ASTAGE;
        const uint8_t *b = a_base + kt * (BK * 2);
#pragma unroll
        for (int q = 0; q < AL; ++q)
            if (q < a_live) {
                if (GATEUP) {
                    uint32_t o = lp[GATEUP ? q : 0];
                    opaque(o);
                    load_lds16(reinterpret_cast<const uint16_t *>(b + (size_t)o * 16), st + (wa + NWA * q) * 1024);
                } else {
                    // h rows in grouped order; rows past the expert's end (all
                    // of a dead group's, with unified roles) repeat its last row
                    const int gr = min(m0 + (wa + NWA * q) * G::RPI + rl, row_end - 1);
                    uint32_t o = (uint32_t)gr * (uint32_t)(I / 8) + a_cs;
                    opaque(o);
                    load_lds16(reinterpret_cast<const uint16_t *>(b + (size_t)o * 16), st + (wa + NWA * q) * 1024);
                }
            }
    };
    auto issue_b_as = [&](int kt, auto aux) __attribute__((always_inline)) {
        uint8_t *st = ring_b + (kt % SB) * BSTAGE;
        const uint8_t *b = b_base + kt * (BK * 2);
#pragma unroll
        for (int q = 0; q < BL; ++q) {
            uint32_t o = b_lane;
            opaque(o);
            load_lds16<decltype(aux)::value>(reinterpret_cast<const uint16_t *>(b + b_row0(q) + o),
                                             st + (wb + NWB * q) * 1024);
        }
    };
    auto issue_b = [&](int kt) __attribute__((always_inline)) {
        if (one_tile) issue_b_as(kt, std::integral_constant<int, kStream>{});
        else issue_b_as(kt, std::integral_constant<int, kDeviceScope>{});
    };

    const int wm = wave / WN, wn = wave % WN;
    const int lrow = lane & 31, lhalf = lane >> 5;
    f32x16_t acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = f32x16_t{};

    // B-tile row of the wave's n-block nb (gate/up pairs share a lane layout)
    auto brow = [&](int nb) {
        return GATEUP ? (nb < NB / 2 ? wn * (TN / 2) + nb * 32 : BN / 2 + wn * (TN / 2) + (nb - NB / 2) * 32)
                      : wn * TN + nb * 32;
    };

    // tile row of this wave's i-th 32-row block
    auto rblk = [&](int i) { return ILV ? (i * WM + wm) * 32 : wm * TM + i * 32; };
    // 32-row blocks of this wave that hold rows of the expert: a tail m-tile
    // of a few rows runs MFMAs and fragment reads on its live blocks only.
    // The count is wave-uniform; the K loop is specialised for each count so
    // every version stays straight-line code.
    const int live_blocks = (row_end - m0 + 31) / 32;
    const int mb_live = __builtin_amdgcn_readfirstlane(
        ILV ? min(MB, max(0, (live_blocks - wm + WM - 1) / WM)) : min(MB, max(0, (row_end - m0 - wm * TM + 31) / 32)));
    // Software-pipelined K loop.  Slot kt % SA of the A ring and kt % SB of
    // the B ring hold stage kt; the stages up to kt+SA-1 / kt+SB-1 are in
    // flight while stage kt is consumed, and the LDS reads of stage kt+1
    // overlap stage kt's MFMAs.
    // ROLE 0: this wave loads both operands (SA == SB); 1: A only; 2: B only
    auto kloop = [&](auto live, auto role_c) __attribute__((always_inline)) {
        constexpr int L = decltype(live)::value;
        constexpr int ROLE = decltype(role_c)::value;
        // a stage of BK is consumed in SUB fragment steps of BKF = FK (16:
        // one MFMA K step, 32: two), so the fragment registers do not grow
        // with BK
        static_assert(FK == 16 || FK == 32, "fragment step of one or two MFMA K steps");
        constexpr int BKF = BK < FK ? BK : FK;
        constexpr int SUB = BK / BKF;
        constexpr int KK = BKF / 16;
        bf16x8_t af[2][KK][MB], bfr[2][KK][NB];
        auto read_frags = [&](int kt, int sub, int buf) __attribute__((always_inline)) {
            const uint8_t *sa = ring_a + (kt % SA) * ASTAGE;
            const uint8_t *sb = ring_b + (kt % SB) * BSTAGE;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                const int c = (sub * KK + kk) * 2 + lhalf;
#pragma unroll
                for (int i = 0; i < L; ++i)
                    af[buf][kk][i] = *reinterpret_cast<const bf16x8_t *>(sa + G::off(rblk(i) + lrow, c));
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    bfr[buf][kk][j] = *reinterpret_cast<const bf16x8_t *>(sb + G::off(brow(j) + lrow, c));
            }
        };
        auto mfmas = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int kk = 0; kk < KK; ++kk)
#pragma unroll
                for (int i = 0; i < L; ++i)
#pragma unroll
                    for (int j = 0; j < NB; ++j)
                        // weights as the first operand: a lane then holds one
                        // activation row and four weight rows in a row (epilogue)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[buf][kk][j], af[buf][kk][i],
                                                                            acc[i][j], 0, 0, 0);
        };
        // prologue: every ring filled, stage 0 landed
        if constexpr (ROLE == 1) {
#pragma unroll
            for (int s0 = 0; s0 < SA; ++s0)
                if (s0 < KT) issue_a(s0);
            wait_vm_rt(min(SA - 1, KT - 1) * a_live);
        } else if constexpr (ROLE == 2) {
#pragma unroll
            for (int s0 = 0; s0 < SB; ++s0)
                if (s0 < KT) issue_b(s0);
            wait_stage<SB + 1, BL>(min(SB - 1, KT - 1));
        } else {
#pragma unroll
            for (int s0 = 0; s0 < SA; ++s0)
                if (s0 < KT) {
                    issue_a(s0);
                    issue_b(s0);
                }
            wait_stage<SA + 1, AL + BL>(min(SA - 1, KT - 1));
        }
        ring_barrier();
        if constexpr (L > 0) read_frags(0, 0, 0);
        // one pipeline step consuming stage kt from fragment buffer CUR:
        // wait for stage kt+1 of this wave's ring(s), synchronise the block
        // (every wave has then also finished reading stage kt, whose
        // fragments are in registers), refill stage kt's slots with stages
        // kt+SA / kt+SB, read stage kt+1's fragments and run stage kt's MFMAs.
        // STEADY: stages kt+1, kt+SA and kt+SB exist (known at compile time).
        // The steady-state loop then has no path around the barrier; such a
        // path joins the loop header, and the compiler's wait analysis would
        // make this stage's MFMAs wait for the next stage's fragment reads.
        auto step = [&](int kt, auto cur_c, auto steady_c) __attribute__((always_inline)) {
            constexpr int CUR0 = decltype(cur_c)::value;
            constexpr bool STEADY = decltype(steady_c)::value;
            // the stage's sub-steps before its last: read the next sub-step's
            // fragments, run this one's MFMAs (no wait: the stage has landed)
#pragma unroll
            for (int sub = 0; sub + 1 < SUB; ++sub) {
                const int cb = CUR0 ^ (sub & 1);
                if constexpr (L > 0) read_frags(kt, sub + 1, cb ^ 1);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (L > 0) mfmas(cb);
                __builtin_amdgcn_sched_barrier(0);
            }
            constexpr int CUR = CUR0 ^ ((SUB - 1) & 1);
            if (STEADY || kt + 1 < KT) {
                if constexpr (ROLE == 1) {
                    if constexpr (STEADY) wait_vm_rt((SA - 2) * a_live);
                    else wait_vm_rt(min(SA - 2, KT - 2 - kt) * a_live);
                } else if constexpr (ROLE == 2) {
                    if constexpr (STEADY) wait_stage<SB, BL>(SB - 2);
                    else wait_stage<SB, BL>(min(SB - 2, KT - 2 - kt));
                } else {
                    if constexpr (STEADY) wait_stage<SA, AL + BL>(SA - 2);
                    else wait_stage<SA, AL + BL>(min(SA - 2, KT - 2 - kt));
                }
                ring_barrier();
                // into stage kt's slots, read out before the barrier
                if constexpr (ROLE == 1) {
                    if (STEADY || kt + SA < KT) issue_a(kt + SA);
                } else if constexpr (ROLE == 2) {
                    if (STEADY || kt + SB < KT) issue_b(kt + SB);
                } else {
                    if (STEADY || kt + SA < KT) {
                        issue_a(kt + SA);
                        issue_b(kt + SA);
                    }
                }
                if constexpr (L > 0) read_frags(kt + 1, 0, CUR ^ 1);
            }
            __builtin_amdgcn_sched_barrier(0);  // keep the next stage's reads ahead of these MFMAs
            if constexpr (L > 0) mfmas(CUR);
            // and keep these MFMAs ahead of the next step's wait and barrier:
            // sunk below them, they would leave the next stage's fragment
            // reads nothing to hide behind before that barrier's lgkmcnt(0)
            __builtin_amdgcn_sched_barrier(0);
        };
        using C0 = std::integral_constant<int, 0>;
        using Steady = std::true_type;
        using Tail = std::false_type;
        // unrolled by two so the fragment buffers are indexed statically
        int kt = 0;
        constexpr int SMAX = SA > SB ? SA : SB;
        // the buffer of a stage's first sub-step alternates with SUB odd
        using CN = std::integral_constant<int, SUB & 1>;
        for (; kt + 1 + SMAX < KT; kt += 2) {
            step(kt, C0{}, Steady{});
            step(kt + 1, CN{}, Steady{});
        }
        for (; kt + 1 < KT; kt += 2) {
            step(kt, C0{}, Tail{});
            step(kt + 1, CN{}, Tail{});
        }
        if (kt < KT) step(kt, C0{}, Tail{});
    };
    // one straight-line K loop per load role (both roles pass the same
    // barriers, once per step) and per live row-block count
    auto run = [&](auto live) __attribute__((always_inline)) {
        if constexpr (SPLIT) {
            if (a_role) kloop(live, std::integral_constant<int, 1>{});
            else kloop(live, std::integral_constant<int, 2>{});
        } else {
            kloop(live, std::integral_constant<int, 0>{});
        }
    };
    if (mb_live >= MB) run(std::integral_constant<int, MB>{});
    else if (mb_live == 0) run(std::integral_constant<int, 0>{});
    else if constexpr (MB >= 2) {
        if (mb_live == 1) run(std::integral_constant<int, 1>{});
        else if constexpr (MB >= 3) {
            if (mb_live == 2) run(std::integral_constant<int, 2>{});
            else if constexpr (MB >= 4) {
                if (mb_live == 3) run(std::integral_constant<int, 3>{});
            }
        }
    }

    // ---- epilogue.  A lane holds row (lane & 31) of each 32x32 block and its
    // columns (r/4)*8 + (lane/32)*4 + r%4, i.e. four groups of four columns.
    // The tile goes through LDS (the ring is free now) and out in 16-byte
    // stores along whole rows, written through.  Against 2-byte stores straight from the
    // accumulators: DeepSeek-V2-Lite shape T=1304 gate/up 167 -> 148 us, down 82 ->
    // 74; Qwen shape T=512 down 76 -> 71, T=4096 down 167 -> 158; whole layers
    // T=512 240 -> 231, T=1304 374 -> 354.  (Row-wise stores without the
    // write-through gave 161 / 82 / 76 / 161.)  A staged row is 16 bytes longer than a multiple of
    // the 256-byte bank line: the 16 rows of a quarter-wave write land in
    // distinct banks.
    constexpr int CO = GATEUP ? BN / 2 : BN;  // output columns of the tile
    constexpr int OB = CO * 2 + 16;           // bytes of a staged row
    static_assert(BM * OB <= SA * ASTAGE + SB * BSTAGE, "staged output fits the ring");
    __syncthreads();  // every wave has read its last stage
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        if (m0 + rblk(i) >= row_end) continue;  // wave-uniform
        uint8_t *const srow = smem + (rblk(i) + lrow) * OB + (wn * (GATEUP ? TN / 2 : TN) + lhalf * 4) * 2;
#pragma unroll
        for (int j = 0; j < (GATEUP ? NB / 2 : NB); ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                uint32_t w[2];
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const int r = q * 4 + p * 2;
                    if constexpr (GATEUP) {
                        const uint32_t g = f2bf2_hw(acc[i][j][r], acc[i][j][r + 1]);
                        const uint32_t u = f2bf2_hw(acc[i][j + NB / 2][r], acc[i][j + NB / 2][r + 1]);
                        const uint32_t a = f2bf2_hw(silu_fast(lo_bf(g)), silu_fast(hi_bf(g)));
                        w[p] = f2bf2_hw(lo_bf(a) * lo_bf(u), hi_bf(a) * hi_bf(u));
                    } else {
                        w[p] = f2bf2_hw(acc[i][j][r], acc[i][j][r + 1]);
                    }
                }
                *reinterpret_cast<uint2 *>(srow + (j * 32 + q * 8) * 2) = make_uint2(w[0], w[1]);
            }
    }
    __syncthreads();
    constexpr int CH = CO / 8;  // 16-byte chunks per row
    const int ldo = GATEUP ? I : H;
    const int chunks = min(BM, row_end - m0) * CH;
    for (int c = tid; c < chunks; c += 64 * NW) {
        const int row = c / CH, ch = c % CH;
        st_through(out + (size_t)(m0 + row) * ldo + n0 + ch * 8,
                   *reinterpret_cast<const uint4 *>(smem + row * OB + ch * 16));
    }
}

template <int BM, int BN, int BK, int WM, int WN, int SA, int SB, bool ILV, bool GATEUP, int OCC, int FK>
__global__ __launch_bounds__(64 * WM * WN, OCC == 1 ? 1 : OCC * WM * WN / 4) void grouped_kernel(
    const uint16_t *__restrict__ a_src, const int32_t *__restrict__ perm_token,
    const int32_t *__restrict__ offsets, const int32_t *__restrict__ sel, int nsel,
    const int32_t *__restrict__ tile_start, const uint16_t *const *__restrict__ slots, int H, int I,
    uint16_t *__restrict__ out, SharedTiles sh) {
    __shared__ __attribute__((aligned(1024))) uint8_t smem[kRingBytes<BM, BN, BK, SA, SB>];
    grouped_tile<BM, BN, BK, WM, WN, SA, SB, ILV, GATEUP, OCC, FK>(smem, a_src, perm_token, offsets, sel, nsel,
                                                                   tile_start, slots, H, I, out, sh);
}

// Gate/up for a mean of about 200..320 rows per expert, where the better tile
// depends on how the rows are spread and only the device knows that: a
// 384-row tile (128 columns) holds most experts of a uniform routing whole,
// where 256-row tiles (256 columns) would read the weights of every expert
// with more than 256 rows twice; a skewed routing has experts of many tiles
// either way, and the wider tile then reads their rows half as often.  Every
// block compares the two m-tile counts of the same order, which the schedule
// launch writes for both heights, and runs one body: 384 rows where they save
// a quarter of the m-tiles or more.  Both halves of the Qwen shape, T=4096:
// uniform (128 tiles against 194) 444 us here, 438 on 384 rows alone and 447 on
// 256; Zipf (178 against 218) 459, 495 and 458: two bodies in one kernel spill
// 110 SGPRs, about 1% where the 384-row one runs (small layer, 94.9 against
// 93.4), and the choice is worth 7% on the skewed routing.
__global__ __launch_bounds__(512, 1) void grouped_gateup_pair_kernel(
    const uint16_t *__restrict__ x, const int32_t *__restrict__ perm_token, const int32_t *__restrict__ offsets,
    const int32_t *__restrict__ sel, int nsel, const int32_t *__restrict__ tile_start_384,
    const int32_t *__restrict__ tile_start_256, const uint16_t *const *__restrict__ slots, int H, int I,
    uint16_t *__restrict__ h_ws, SharedTiles sh) {
    constexpr int B384 = kRingBytes<384, 128, 64, 2, 4>, B256 = kRingBytes<256, 256, 64, 2, 3>;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[B384 > B256 ? B384 : B256];
    const int m384 = tile_start_384[nsel], m256 = tile_start_256[nsel];
    if (4 * m384 <= 3 * m256)
        grouped_tile<384, 128, 64, 4, 2, 2, 4, true, true, 1, 32>(smem, x, perm_token, offsets, sel, nsel,
                                                                  tile_start_384, slots, H, I, h_ws, sh);
    else
        grouped_tile<256, 256, 64, 2, 4, 2, 3, true, true, 1, 16>(smem, x, perm_token, offsets, sel, nsel,
                                                                  tile_start_256, slots, H, I, h_ws, sh);
}

// Everything a grouped launch takes beside its tile configuration.
struct GroupedArgs {
    const uint16_t *x;
    const int32_t *perm_token, *offsets, *sel;
    int nsel;
    const int32_t *tile_start;
    int max_tiles;
    const uint16_t *const *slots;
    int H, I;
    uint16_t *h_ws, *y;
    SharedTiles sh;
    hipStream_t s;
};

// Blocks of a launch: the shared tiles', then every (m-tile, n-tile) the bound
// allows, each a multiple of 8 so each XCD's contiguous piece of a tile range
// has blocks.
static unsigned grouped_grid(const GroupedArgs &a, int max_tiles, int BM, int nt, int nt_shared) {
    const size_t shared = a.sh.slot ? (size_t)((a.sh.T + BM - 1) / BM) * (size_t)nt_shared : 0;
    return (unsigned)((shared + 7) / 8 * 8 + ((size_t)max_tiles * (size_t)nt + 7) / 8 * 8);
}

// phase: 1 = gate/up only, 2 = down only, 3 = both
// PH: the phases (1 gate/up, 2 down) this tile configuration serves
template <int BM, int BN, int BK, int WM, int WN, int SA, int SB, bool ILV = false, int PH = 3, int OCC = 1,
          int FK = 32>
int launch_grouped(int phase, const GroupedArgs &a) {
    static_assert(BK == 64, "grouped_check: H and I divide by 64");
    if constexpr ((PH & 1) != 0) if (phase & 1) {
        grouped_kernel<BM, BN, BK, WM, WN, SA, SB, ILV, true, OCC, FK>
            <<<grouped_grid(a, a.max_tiles, BM, a.I / (BN / 2), a.sh.I / (BN / 2)), 64 * WM * WN, 0, a.s>>>(
                a.x, a.perm_token, a.offsets, a.sel, a.nsel, a.tile_start, a.slots, a.H, a.I, a.h_ws, a.sh);
        int rc = check_launch("grouped_kernel<gateup>");
        if (rc) return rc;
    }
    if constexpr ((PH & 2) != 0) if (phase & 2) {
        grouped_kernel<BM, BN, BK, WM, WN, SA, SB, ILV, false, OCC, FK>
            <<<grouped_grid(a, a.max_tiles, BM, a.H / BN, a.H / BN), 64 * WM * WN, 0, a.s>>>(
                a.h_ws, nullptr, a.offsets, a.sel, a.nsel, a.tile_start, a.slots, a.H, a.I, a.y, a.sh);
        return check_launch("grouped_kernel<down>");
    }
    return kOk;
}

// Every check of a call, before anything is launched.  A row tile of 384 takes
// 128 columns, the others 256 (also where a narrower form of the tile runs:
// which shapes are taken does not depend on the number of experts).
static int grouped_check(int phase, int block_m, const GroupedArgs &a) {
    if (((phase & 1) && (!a.x || !a.perm_token)) || !a.offsets || !a.sel || !a.tile_start || !a.slots || !a.h_ws ||
        ((phase & 2) && !a.y))
        return fail(kEInval, "grouped: null pointer");
    if (a.nsel < 1 || a.max_tiles < 1) return fail(kEInval, "grouped: need nsel >= 1 and max_tiles >= 1");
    if (a.max_tiles > (1 << 22)) return fail(kEInval, "grouped: max_tiles too large");
    if (block_m != 32 && block_m != 64 && block_m != 128 && block_m != 256 && block_m != 384)
        return fail(kEInval, "grouped: block_m must be 32, 64, 128, 256 or 384");
    const int cols = block_m == 384 ? 128 : 256;
    if (a.H < cols || a.H % cols || a.I < cols / 2 || a.I % (cols / 2))
        return fail(kEInval, "grouped: need H % 256 == 0 and I % 128 == 0 (block_m 384: H % 128, I % 64)");
    if (a.sh.slot && (a.sh.I < cols / 2 || a.sh.I % (cols / 2) || a.sh.T < 1 || !a.sh.h || !a.sh.y))
        return fail(kEInval, "grouped: bad shared arguments (shared I % 128 == 0; block_m 384: % 64)");
    return kOk;
}

// Whether `tiles` equal tiles on `slots` workgroups end in a round that fills
// at most half of them, early enough (below four rounds) to cost a good part
// of the launch.
static bool sparse_last_round(int tiles, int slots) {
    const int rest = tiles % slots;
    return tiles > slots && tiles < 4 * slots && rest != 0 && 2 * rest <= slots;
}

// The launches of a checked call.
static int grouped_phase(int phase, int block_m, const GroupedArgs &a) {
    int rc = kOk;
    switch (block_m) {
    case 32:
        // down (K = I, a short K loop): two workgroups of 128 columns per CU, so
        // that one's ring fill and epilogue overlap the other's loads (T=201:
        // 71 -> 67 us, T=17: 46.8 -> 44.5); gate/up is faster on 256 columns
        // and a CU of its own (T=201: 128 us against 136 at two per CU)
        if (phase & 1) rc = launch_grouped<32, 256, 64, 1, 4, 4, 4, false, 1>(1, a);
        if (rc == kOk && (phase & 2)) rc = launch_grouped<32, 128, 64, 1, 4, 4, 4, false, 2, 2>(2, a);
        return rc;
    case 64:
        // gate/up: split load roles, 3 + 4 stages, one workgroup per CU; down
        // (K = I, a short K loop): every wave loads both operands, 2 + 2
        // stages, two workgroups per CU (T=512: 79.6 against 85.3 us)
        // Half-width tiles, two workgroups per CU, where one m-tile per expert of
        // the full width ends in a sparse round on 256 CUs (96 experts of I = 384
        // are 288 tiles: T=201 52 -> 45 us, T=450 54 -> 47; H = 1536 down 27 ->
        // 25; 87 of the Qwen shape's experts, 32 rows each, 107 -> 99, 106 of
        // them 116 -> 110).  With full rounds they read alike (128 of them 131
        // against 133, down 71 against 75) or slower (DeepSeek-V2-Lite shape T=300
        // 125 against 127).
        if (phase & 1)
            rc = sparse_last_round(a.nsel * (a.I / 128), 256) ? launch_grouped<64, 128, 64, 2, 2, 3, 3, false, 1, 2>(1, a)
                                                              : launch_grouped<64, 256, 64, 2, 4, 3, 4, false, 1>(1, a);
        if (rc == kOk && (phase & 2))
            rc = sparse_last_round(a.nsel * (a.H / 256), 512) ? launch_grouped<64, 128, 64, 2, 2, 3, 3, false, 2, 2>(2, a)
                                                              : launch_grouped<64, 256, 64, 2, 4, 2, 2, false, 2, 2>(2, a);
        return rc;
    case 128:
        return launch_grouped<128, 256, 64, 2, 4, 3, 3>(phase, a);
    case 256:
        // 128-byte row pieces (BK 64) halve the L2 requests of the 64-byte
        // ones; each CU keeps about 64 requests in flight, so the bytes per
        // request set its fill rate.  Fragments are read one MFMA K step (16)
        // ahead, which keeps the tile within 256 VGPRs without spills, and
        // split load roles with 2 + 3 stages fill the 160 KB of LDS
        // (T=4096, Zipf routing: gate/up 338 -> 299 us, down 199 -> 173 us;
        // uniform: down 190 -> 161 us; bit-identical)
        // 32-row blocks dealt to the two wave rows in turn: an expert of fewer
        // rows than the tile keeps both busy (T=2048, 128 rows each: gate/up
        // 163 -> 153 us, down 96 -> 90; T=4096 Zipf down 173 -> 162)
        return launch_grouped<256, 256, 64, 2, 4, 2, 3, true, 3, 1, 16>(phase, a);
    default:  // 384
        return launch_grouped<384, 128, 64, 4, 2, 2, 4, true>(phase, a);
    }
}

static int grouped_entry(int phase, const void *x, const int32_t *perm_token, const int32_t *offsets,
                         const int32_t *sel, int nsel, const int32_t *tile_start, int max_tiles, int block_m,
                         const void *const *slots, int H, int I, void *h_ws, void *y, void *stream) {
    const GroupedArgs a{(const uint16_t *)x, perm_token, offsets, sel, nsel, tile_start, max_tiles,
                        (const uint16_t *const *)slots, H, I, (uint16_t *)h_ws, (uint16_t *)y,
                        SharedTiles{nullptr, 0, 0, nullptr, nullptr}, reinterpret_cast<hipStream_t>(stream)};
    const int rc = grouped_check(phase, block_m, a);
    return rc != kOk ? rc : grouped_phase(phase, block_m, a);
}

}  // namespace pd

using namespace pd;

// The row tile should cover a typical expert in one tile (weights are then
// read once per expert and n-tile); 32 only for very thin experts.
PD_API int pdscope_grouped_block_m(int rows_hint) {
    if (rows_hint <= 16) return 32;
    // whole Qwen-shaped layers (pack + gate/up + down + merge), uniform
    // routing, back to back: 24..40 mean rows run fastest on 64-row tiles,
    // 48..96 on 128-row tiles (64 rows: 271 against 292 us), 112 and above on
    // the 256-row tile (112: 309 against 320 us; the DeepSeek-V2-Lite mixed
    // batch, 122 mean rows of 17 MB experts: 332 against 355 us)
    if (rows_hint <= 44) return 64;
    if (rows_hint <= 104) return 128;
    if (rows_hint <= 192) return 256;
    // one 384-row tile holds an expert of the typical 200..320 rows (no
    // tail tile re-reading its weights); beyond that 256x256 tiles read the
    // activation rows fewer times
    if (rows_hint <= 320) return 384;
    return 256;
}

// The row tile for a mean of rows_hint rows over nsel experts of intermediate
// I: pdscope_grouped_block_m, except that thin experts take the 64-row tile
// where its half-width form fills the chip better (see block_m 64 above).  That
// counts a tile for every expert, so it needs two rows each: at a mean of one,
// about 0.63 of them have rows (96 experts of I = 384 are 180 tiles, no second
// round at all).  Whole layers of that shape on 32 and 64 rows: T=16 57.8 and
// 60.2 us, T=24 64.9 and 65.3, T=32 (two rows each) 71.3 and 70.6, T=40 86.8 and
// 80.7, T=200 93.1 and 86.5.
PD_API int pdscope_grouped_block_m_shape(int rows_hint, int nsel, int I) {
    const int bm = pdscope_grouped_block_m(rows_hint);
    return bm == 32 && rows_hint >= 2 && sparse_last_round(nsel * (I / 128), 256) ? 64 : bm;
}

PD_API int pdscope_grouped_block_m_max(int mean_rows, int max_rows) {
    const int bm = pdscope_grouped_block_m(mean_rows);
    return bm == 384 && max_rows > 768 ? 256 : bm;
}

PD_API int pdscope_swiglu_grouped(const void *x, const int32_t *perm_token, const int32_t *offsets,
                                  const int32_t *sel, int nsel, const int32_t *tile_start, int max_tiles,
                                  int block_m, const void *const *slots, int H, int I, void *h_ws, void *y,
                                  void *stream) {
    return grouped_entry(3, x, perm_token, offsets, sel, nsel, tile_start, max_tiles, block_m, slots, H, I, h_ws, y,
                         stream);
}

PD_API int pdscope_swiglu_grouped_gateup(const void *x, const int32_t *perm_token, const int32_t *offsets,
                                         const int32_t *sel, int nsel, const int32_t *tile_start, int max_tiles,
                                         int block_m, const void *const *slots, int H, int I, void *h_ws,
                                         void *stream) {
    return grouped_entry(1, x, perm_token, offsets, sel, nsel, tile_start, max_tiles, block_m, slots, H, I, h_ws,
                         nullptr, stream);
}

PD_API int pdscope_swiglu_grouped_layer(const void *x, const int32_t *perm_token, const int32_t *offsets,
                                        const int32_t *sel, int nsel, const int32_t *tile_start, int max_tiles,
                                        int block_m, const int32_t *tile_start_down, int max_tiles_down,
                                        int block_m_down, const void *const *slots, int H, int I, void *h_ws, void *y,
                                        int T, const void *const *shared_slot, int shared_I, void *h_shared,
                                        void *y_shared, void *stream) {
    const SharedTiles sh = {(const uint16_t *const *)shared_slot, shared_slot ? shared_I : 0, T, (uint16_t *)h_shared,
                            (uint16_t *)y_shared};
    GroupedArgs a{(const uint16_t *)x, perm_token, offsets, sel, nsel, tile_start, max_tiles,
                  (const uint16_t *const *)slots, H, I, (uint16_t *)h_ws, (uint16_t *)y, sh,
                  reinterpret_cast<hipStream_t>(stream)};
    GroupedArgs d = a;
    d.tile_start = tile_start_down;
    d.max_tiles = max_tiles_down;
    int rc = grouped_check(1, block_m, a);
    if (rc == kOk) rc = grouped_check(2, block_m_down, d);
    if (rc != kOk) return rc;
    if (block_m != 384 || block_m_down != 256) {
        rc = grouped_phase(1, block_m, a);
        return rc != kOk ? rc : grouped_phase(2, block_m_down, d);
    }
    const unsigned grid = std::max(grouped_grid(a, max_tiles, 384, I / 64, sh.I / 64),
                                   grouped_grid(d, max_tiles_down, 256, I / 128, sh.I / 128));
    grouped_gateup_pair_kernel<<<grid, 512, 0, a.s>>>(a.x, perm_token, offsets, sel, nsel, tile_start, tile_start_down,
                                                      a.slots, H, I, a.h_ws, sh);
    rc = check_launch("grouped_gateup_pair_kernel");
    return rc != kOk ? rc : grouped_phase(2, 256, d);
}

PD_API int pdscope_swiglu_grouped_down(const void *h_ws, const int32_t *offsets, const int32_t *sel, int nsel,
                                       const int32_t *tile_start, int max_tiles, int block_m,
                                       const void *const *slots, int H, int I, void *y, void *stream) {
    return grouped_entry(2, nullptr, nullptr, offsets, sel, nsel, tile_start, max_tiles, block_m, slots, H, I,
                         const_cast<void *>(h_ws), y, stream);
}
