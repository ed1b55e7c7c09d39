// The wide matrix-core kernel: matmul of a K-quant weight with batches (Q4_K of more than 32 tokens,
// Q6_K of more than 16 and fewer on weights without a K cut; the launchers of the narrow kernels say which),
// and of the expert groups of a routed layer.  One workgroup per (block of weight rows,
// column of up to 128 tokens); gemm_q6k_wide.hip and gemm_q4k_wide.hip supply the formats.
//
// A wave owns ONE 16-row tile and all tokens of its workgroup's column: what a super-block of
// weights costs to unpack into int8 operands is paid once for up to eight token groups of 16.
//
// Everything a step reads -- the super-block of weights of every wave's tile, the activation slab
// (256 values of every token of the column), now and then the activation scales -- goes from memory
// to LDS without passing through registers (global_load_lds).  A lane's register loads of a weight
// tile would touch 16 rows per instruction and keep the address unit busy for 31 - 39 cycles each,
// more than the bytes take; here every request reads whole lines.  LDS is written at consecutive addresses, 16
// bytes per lane, so bank conflicts are kept down by what each lane FETCHES (a tenth of the LDS cycles are left on Q4_K,
// 14336 x 4096 at 512 tokens): 16-byte slot p of
// token t holds piece p ^ (t % 16) of its 256 values (the weights likewise).  A reader applies the
// same exclusive-or.
//
// Results are the matvec's bits: the exact integers of a super-block, then its f32 steps, in order;
// where the matvec cuts K for a weight shape the same parts are summed left to right here, on KS = 2
// groups of waves (each walking half of the parts) or inside the lane (SPLIT).
#pragma once

#include <algorithm>
#include <atomic>
#include <cmath>
#include <string>

#include "cml_device.hpp"
#include "cml_host.hpp"

#pragma clang fp contract(off)

namespace cml {

typedef int v4i_w __attribute__((ext_vector_type(4)));
typedef float v4f_w __attribute__((ext_vector_type(4)));
typedef float v16f_w __attribute__((ext_vector_type(16)));
typedef _Float16 v4h_w __attribute__((ext_vector_type(4)));

// One wave's 1 KB: lane l's 16 bytes at base + off (off per lane) to LDS byte lds_byte + 16 * l (lds_byte wave-uniform).
// Written as assembly because the compiler, which cannot tell which LDS bytes such a load will
// write, puts a wait for all of them in front of every later LDS read; here the caller waits
// (wide_wait) where the data is first needed.  The compiler does not look inside for the wait states the hardware wants
// either: five between a vector instruction that writes a scalar register (v_readlane: a base that was spilled) and a memory
// instruction that addresses through it, one between a write of m0 and an instruction that addresses LDS through it.
// The scalar move of the base is both: the hardware holds it back until the base is written, and it stands behind m0.
__device__ __forceinline__ void wide_dma16(uint32_t lds_byte, const void *base, uint32_t off) {
    const void *at;
    asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0" : "=&s"(at) : "s"(lds_byte), "v"(off), "s"(base) : "memory", "m0");
}
// The same for bytes that are read once (non-temporal: 768 MB in long runs 129 us plain, 115 so).
__device__ __forceinline__ void wide_dma16_once(uint32_t lds_byte, const void *base, uint32_t off) {
    const void *at;
    asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dwordx4 %2, %0 nt" : "=&s"(at) : "s"(lds_byte), "v"(off), "s"(base) : "memory", "m0");
}
// The same with 4 bytes per lane.
__device__ __forceinline__ void wide_dma4(uint32_t lds_byte, const void *base, uint32_t off) {
    const void *at;
    asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, %3\n\tglobal_load_lds_dword %2, %0" : "=&s"(at) : "s"(lds_byte), "v"(off), "s"(base) : "memory", "m0");
}
template <bool ONCE>
__device__ __forceinline__ void wide_dma16_hint(uint32_t lds_byte, const void *base, uint32_t off) {
    if constexpr (ONCE) wide_dma16_once(lds_byte, base, off);
    else wide_dma16(lds_byte, base, off);
}
// Waits until at most OUT of the wave's vector-memory operations are outstanding (loads complete in order).
template <int OUT>
__device__ __forceinline__ void wide_wait() {
    static_assert(OUT < 64, "six bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(OUT) : "memory");
}
// Workgroup barrier after this wave's LDS operations (__syncthreads would also wait for every load in flight).
__device__ __forceinline__ void wide_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Which weights are requested past the 256 MB last-level cache: those of 96 MB and more.  A weight of that size is used once in a pass over a model, whose other weights have taken its
// place when it is used again (plain / so, 600 MB of other weights between, us: Q8_0 32000 x 4096, 139 MB, at 8 tokens 32.5 / 29.4, 128256 x 2048, 279 MB, at 16 57.4 / 54.7; Q4_0
// 128256 x 3072, 222 MB, at 16 57.3 / 55.8; expert layers, three tensors of the size each, 1 GB of other layers between: Q4_K 8 x 4096 / 14336, 264 MB, at 64 / 128 / 512 tokens
// 229 / 216, 282 / 270, 679 / 668, 3072 / 8192, 113 MB, at 128 145 / 143; Q8_0 8 x 4096 / 4096, 143 MB, at 16 / 64 124 / 111, 115 / 107).  Where nothing is used in between, the cache holds
// weights of up to 256 MB and the hint costs: the two plain ones above back to back 26.4 / 32.0 and 43.9 / 58.5.  Smaller weights stay: Q4_K 1536 / 6144, 42 MB, one layer over and over, at 128
// 77 / 81.  That a K-quant group of more than a column reads its rows again costs nothing (a column holds up to 128 assignments); with columns of 16 and 32 it does: Q8_0
// 8 x 4096 / 4096 at 256 239 / 274, all assignments on few experts 267 / 315.
inline bool wide_reads_once(const cml_weight *w) {
    const int64_t block = w->fmt == CML_Q8_0 ? 34 : w->fmt == CML_Q4_0 ? 18 : w->fmt == CML_Q4_K ? 144 : 210;
    const int forced = env_int("CAMELID_HIP_WIDE_ONCE", -1);  // 0 = never, 1 = always
    return forced >= 0 ? forced != 0 : w->rows * w->nb * block >= 96ll << 20;
}

// LDS byte address of a shared-memory pointer.
__device__ __forceinline__ uint32_t lds_address(const void *p) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void *)p));
}

// Workgroup id -> (row block, token column).  Consecutive ids go to the eight XCDs in turn; the columns of one row
// block are given to ONE XCD, one after the other, so that its rows of the weight come through that XCD's L2 once.
// The grid is padded to whole rounds of eight row blocks: row blocks past the end return false.
__device__ __forceinline__ bool wide_block(int id, int n_row_blocks, int n_cols, int &row_block, int &col) {
    const int j = id >> 3, r = j / n_cols;
    row_block = r * 8 + (id & 7);
    col = j - r * n_cols;
    return row_block < n_row_blocks;
}
inline unsigned wide_grid(int64_t n_row_blocks, int64_t n_cols) { return static_cast<unsigned>((n_row_blocks + 7) / 8 * 8 * n_cols); }

template <class F>
struct WideArgs {
    typename F::Weight w;
    int rows, n_sb;     // rows of one band; super-blocks per row
    int row_skip;       // leading rows of the first tile that precede this weight view (0..15)
    int n_tiles;        // 16-row tiles of one band
    int n_row_blocks;   // of both weights of a pair launch
    int n_cols;         // token columns in the grid (expert groups: one, which walks them all)
    int ksplit;         // association to reproduce (the matvec kernel's K cut)
    const int8_t *q;    // [n_tokens][n_sb*256]
    const float *yd;    // [n_tokens][n_sb]
    float *out;         // [n_tokens][rows]
    int n_tokens;       // plain: activation rows; grouped: the most assignments one group can hold
    // Grouped call (mixture of experts): blockIdx.y -> group e (through group_ids when set; -1 = unused slot), which owns
    // the weight band of rows [e*rows, (e+1)*rows) and the assignments [group_offsets[e], group_offsets[e+1]); assignment
    // j reads activation row group_rows[j] (j itself when null) and writes output row j.
    const int32_t *group_offsets;
    const int32_t *group_rows;
    const int32_t *group_ids;
    // Pair launch (grouped calls): a second stacked weight of the same shape against the same activations, written to out2;
    // its row blocks follow the first's.
    typename F::Weight w2;
    float *out2;
};

// LDS layout of one workgroup.
template <class F, int G, int WAVES, int KS>
struct WideLds {
    static constexpr int NTOK = 16 * G;
    static constexpr int kSlab = NTOK * 256;                   // one activation slab, pieces exclusive-ored
    static constexpr int kRuns = F::kRunSums ? NTOK * 32 : 0;  // the sums of its 16-value runs, f16
    static constexpr int kYd = (NTOK + 63) / 64 * 256;         // activation scales of one step
    // weights: one super-block of every wave's tile, two steps ahead where that fits
    static constexpr int kW = WAVES * F::kTileBytes;
    static constexpr int kBase = 2 * KS * (kSlab + kRuns + kYd);
    // (two workgroups per compute unit before two steps ahead)
    static constexpr int kHalf = 80 * 1024;
    static constexpr int WS = kBase + 2 * kW <= kHalf ? 2 : kBase + kW <= kHalf ? 1 : kBase + 2 * kW <= 2 * kHalf ? 2 : 1;
    static constexpr int kTotal = kBase + WS * kW;
};

// F: the weight format.  G: token groups of 16 per column.  WAVES: waves per workgroup, WAVES / KS row tiles.
// KS: groups of waves the K parts are shared over (1 or 2).  SPLIT: K parts are closed inside the lane.
// GROUPED: expert groups (token groups past a group's last assignment are skipped, rows are gathered).  ONCE: wide_reads_once.
template <class F, int G, int WAVES, int KS, bool SPLIT, bool GROUPED, bool ONCE>
__global__ __launch_bounds__(64 * WAVES, GROUPED && WAVES == 4 && G <= 3 ? 3 : 2) void gemm_wide_kernel(WideArgs<F> a) {
    typedef WideLds<F, G, WAVES, KS> L;
    constexpr int NTOK = L::NTOK, RT = WAVES / KS, WS = L::WS;
    constexpr int kThreads = 64 * WAVES, kRowsPass = kThreads / 16;        // tokens fetched per pass of the workgroup
    constexpr int kPer = (NTOK + kRowsPass - 1) / kRowsPass;               // passes per slab
    static_assert(KS == 1 || (KS == 2 && !GROUPED), "K parts");
    // A matrix instruction forms the products of the activation's and the weight's scales; not where three waves share a SIMD's registers (expert groups).
    constexpr bool kProducts = F::kScaleGroups > 0 && !GROUPED;
    constexpr int kPair = kProducts ? F::kScaleGroups : 1;
    extern __shared__ uint4 smem[];
    uint8_t *slabs = reinterpret_cast<uint8_t *>(smem);                      // [2][KS][NTOK][256]
    uint8_t *runs = slabs + 2 * KS * L::kSlab;                               // [2][KS][NTOK][16] f16
    constexpr int kYdAt = 2 * KS * (L::kSlab + L::kRuns);
    const float *yds = reinterpret_cast<const float *>(slabs + kYdAt);       // [2][KS][NTOK rounded up to 64]
    constexpr int kWAt = kYdAt + 2 * KS * L::kYd;
    const uint8_t *wbuf = slabs + kWAt;                                      // [WS][WAVES][kTileBytes]

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int n_sb = a.n_sb;
    const int n = lane & 15, kq = lane >> 4;
    int row_block, col;
    if (!wide_block(blockIdx.x, a.n_row_blocks, a.n_cols, row_block, col)) return;
    const int64_t band = GROUPED ? (a.group_ids ? a.group_ids[blockIdx.y] : static_cast<int>(blockIdx.y)) : 0;
    if (band < 0) return;
    const int a0 = GROUPED ? a.group_offsets[band] : 0;
    const int n_assign = GROUPED ? a.group_offsets[band + 1] - a0 : a.n_tokens;
    // Expert groups: one workgroup walks all columns of its group (workgroups of a column of their own would mostly find
    // it empty, each after two dependent loads: with two columns 282 us per Mixtral-shaped layer of 64 tokens, 200 so).
    for (;; col++) {
        const int tok0 = col * NTOK;
        if (tok0 >= n_assign) return;  // the whole workgroup leaves
        const int n_here = min(NTOK, n_assign - tok0);
        const int n_blk = (a.n_tiles + RT - 1) / RT;
        const bool second = GROUPED && row_block >= n_blk;
        const int ks = KS == 2 ? wave / RT : 0;
        const int tile = (row_block - (second ? n_blk : 0)) * RT + (KS == 2 ? wave - ks * RT : wave);
        // this wave group's part of K
        const int k_mid = KS == 2 ? (a.ksplit / 2) * n_sb / a.ksplit : n_sb;
        const int s_begin = ks ? k_mid : 0, n_loc = ks ? n_sb - k_mid : k_mid;
        const int n_max = KS == 2 ? max(k_mid, n_sb - k_mid) : n_sb;

        auto act_row = [&](int t) __attribute__((always_inline)) -> uint32_t {  // (tokens past the end repeat the last one)
            const int j = min(t, n_here - 1);
            return static_cast<uint32_t>(GROUPED ? (a.group_rows ? a.group_rows[a0 + tok0 + j] : a0 + tok0 + j) : j);
        };
        const uint32_t lds0 = lds_address(smem);
        // Activation: thread tid fetches slot tid % 16 of tokens tid / 16 + kRowsPass * k; a wave whose tokens lie past the column does not fetch.
        const int t16 = tid >> 4, piece = (tid & 15) ^ (t16 & 15);
        const uint32_t row_bytes = n_sb * 256u;
        const int8_t *q_base = a.q + (GROUPED ? 0 : static_cast<int64_t>(tok0) * row_bytes);
        uint32_t src[kPer];
#pragma unroll
        for (int k = 0; k < kPer; k++) src[k] = act_row(t16 + kRowsPass * k) * row_bytes + piece * 16;
        auto fetch = [&](int loc, int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int kp = 0; kp < KS; kp++) {
                const int sb = min((kp ? k_mid : 0) + loc, n_sb - 1);
#pragma unroll
                for (int k = 0; k < kPer; k++)
                    if ((kPer * kRowsPass == NTOK || 4 * wave + kRowsPass * k < NTOK) && (!GROUPED || 4 * wave + kRowsPass * k < n_here))
                        wide_dma16(lds0 + (buf * KS + kp) * L::kSlab + k * (16 * kThreads) + wave * 1024, q_base + sb * 256, src[k]);
            }
        };
        // Scales: wave w of the first KS * NTOK / 64 fetches those of tokens 64 (w / KS) + lane for part w % KS.
        const bool yd_wave = wave < KS * (L::kYd / 256);
        const int ykp = wave % KS, yt = wave / KS * 64;
        const float *yd_base = a.yd + (GROUPED ? 0 : static_cast<int64_t>(tok0) * n_sb);
        const uint32_t yd_src = act_row(yt + lane) * n_sb * 4u;
        auto fetch_yd = [&](int loc, int buf) __attribute__((always_inline)) {
            if (yd_wave) wide_dma4(lds0 + kYdAt + (buf * KS + ykp) * L::kYd + yt * 4, yd_base + min((ykp ? k_mid : 0) + loc, n_sb - 1), yd_src);
        };
        // What is derived from a slab: after its wait a lane may read what it has fetched itself.
        auto finish = [&](int buf) __attribute__((always_inline)) {
            if constexpr (F::kRunSums) {
#pragma unroll
                for (int kp = 0; kp < KS; kp++)
#pragma unroll
                    for (int k = 0; k < kPer; k++)
                        if ((kPer * kRowsPass == NTOK || 4 * wave + kRowsPass * k < NTOK) && (!GROUPED || 4 * wave + kRowsPass * k < n_here)) {
                            const uint4 v = *reinterpret_cast<const uint4 *>(slabs + (buf * KS + kp) * L::kSlab + (tid + kThreads * k) * 16);
                            *reinterpret_cast<_Float16 *>(runs + (buf * KS + kp) * L::kRuns + (t16 + kRowsPass * k) * 32 + piece * 2) =
                                static_cast<_Float16>(static_cast<short>(bytesum16(v)));  // (|sum| <= 2048: exact)
                        }
            }
        };

        const F fmt(second ? a.w2 : a.w, band, a.rows, min(tile, a.n_tiles - 1), lane);
        const uint32_t w_lds = lds0 + kWAt + wave * F::kTileBytes;
        const uint8_t *w_mine = wbuf + wave * F::kTileBytes;
        auto fetch_w = [&](int loc, int slot) __attribute__((always_inline)) { fmt.template fetch<ONCE>(w_lds + slot * L::kW, min(s_begin + loc, n_sb - 1)); };

        // A operand of step c: piece (lane's) ^ (step's) of token n
        uint32_t a_addr[4];
#pragma unroll
        for (int c = 0; c < 4; c++) a_addr[c] = n * 256 + ((F::lane_piece(kq) ^ n ^ F::step_piece(c)) << 4);

        fetch_yd(0, 0);
        fetch(0, 0);
        fetch_w(0, 0);
        if constexpr (WS == 2) fetch_w(1, 1);
        typename F::Raw raw;
        wide_wait<(WS - 1) * F::kFetches>();
        fmt.read(raw, w_mine, s_begin);
        finish(0);
        wide_barrier();

        float acc[G][4], total[SPLIT ? G : 1][4];
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[g][j] = 0.0f;
        // K parts closed inside the lane: of the whole row, or of this wave group's half of the parts
        const int part0 = ks ? a.ksplit / 2 : 0;
        int part = 0;
        int next_cut = SPLIT ? (part0 + 1) * n_sb / a.ksplit : 0;

        auto step = [&](int loc, int buf) __attribute__((always_inline)) {
            if constexpr (SPLIT) {
                if (s_begin + loc == next_cut && loc < n_loc) {  // the matvec kernel's K-split point: close the partial chain
#pragma unroll
                    for (int g = 0; g < G; g++)
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            total[g][j] = part == 0 ? acc[g][j] : total[g][j] + acc[g][j];
                            acc[g][j] = 0.0f;
                        }
                    part++;
                    next_cut = (part0 + part + 1) * n_sb / a.ksplit;
                }
            }
            // Requests: the next slab (and scales), then weights WS steps ahead, which alone may be outstanding at the end of the step.
            // (Past the end the last super-block is fetched again: the number of requests in flight stays the same.)
            fetch_yd(loc + 1, buf ^ 1);
            fetch(loc + 1, buf ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            typename F::Operands ops;
            fmt.unpack(raw, ops);
            __builtin_amdgcn_sched_barrier(0);
            fetch_w(loc + WS, WS == 2 ? buf : 0);  // (its slot was read into registers a step ago)
            __builtin_amdgcn_sched_barrier(0);
            const uint8_t *slab = slabs + (buf * KS + ks) * L::kSlab;
            const uint8_t *run = runs + (buf * KS + ks) * L::kRuns + n * 32 + kq * 8;
            const float *ydp = yds + (buf * KS + ks) * (L::kYd / 4) + (kProducts ? 16 * (lane / (64 / kPair)) + n : 4 * kq);
            if (KS == 1 || loc < n_loc) {
                // Software pipeline over the token groups: while the matrix cores work on group g, the operands of group g + 1
                // are read from LDS and the f32 steps of group g - 1 run.
                v4i_w av[2][4];
                v4h_w rs[2];
                float4 yd4[kProducts ? 1 : 3];
                float ya[kProducts ? 2 : 1];
                v16f_w scale[kProducts ? 2 : 1];  // products of the scales of two token groups and of the weight's, all cells of a tile
                typename F::Sums sums[2];
                auto read = [&](int g) __attribute__((always_inline)) {
#pragma unroll
                    for (int c = 0; c < 4; c++) av[g & 1][c] = *reinterpret_cast<const v4i_w *>(slab + a_addr[c] + g * 4096);
                    if constexpr (F::kRunSums) rs[g & 1] = *reinterpret_cast<const v4h_w *>(run + g * 512);
                    if constexpr (!kProducts) yd4[g % 3] = *reinterpret_cast<const float4 *>(ydp + g * 16);
                    else if (g % kPair == 0) ya[g / kPair & 1] = ydp[g * 16];
                };
                auto chain = [&](int g) __attribute__((always_inline)) {
                    if constexpr (kProducts) {
                        fmt.chain(sums[g & 1], scale[g / kPair & 1], g % kPair, acc[g]);
                    } else {
                        const float yv[4] = {yd4[g % 3].x, yd4[g % 3].y, yd4[g % 3].z, yd4[g % 3].w};
                        fmt.chain(sums[g & 1], yv, ops, acc[g]);
                    }
                    // (left alone, the compiler sinks the chains of all steps to the store and keeps every operand alive)
#pragma unroll
                    for (int j = 0; j < 4; j++) asm volatile("" : "+v"(acc[g][j]));
                };
                read(0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int g = 0; g < G; g++) {
                    if (!GROUPED || 16 * g < n_here) {
                        if (g + 1 < G) read(g + 1);
                        fmt.contract(ops, av[g & 1], rs[g & 1], sums[g & 1]);
                        if constexpr (kProducts)
                            if (g % kPair == 0) scale[g / kPair & 1] = __builtin_amdgcn_mfma_f32_16x16x1f32(ya[g / kPair & 1], ops.scale, v16f_w{}, 0, 0, 0);
                        if (g > 0) chain(g - 1);
                        __builtin_amdgcn_sched_group_barrier(0x100, F::kRunSums ? 6 : 5, 0);
#pragma unroll
                        for (int m = 0; m < F::kMfma; m++) {
                            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x2, F::kScaleGroups == 0 || kProducts ? 2 : 3, 0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                        if (g == G - 1 || (GROUPED && 16 * (g + 1) >= n_here)) chain(g);
                    }
                }
            }
            wide_wait<(WS - 1) * F::kFetches>();
            fmt.read(raw, w_mine + (WS == 2 ? (buf ^ 1) * L::kW : 0), min(s_begin + loc + 1, n_sb - 1));
            finish(buf ^ 1);
            wide_barrier();
        };
        // (two steps per round: buffer addresses are known at compile time)
        int loc = 0;
        for (; loc + 2 <= n_max; loc += 2) {
            step(loc, 0);
            step(loc + 1, 1);
        }
        if (loc < n_max) step(loc, 0);
        wide_wait<0>();  // (nothing may still be on its way into LDS that is reused or given back)

        if constexpr (KS == 2) {
            // The second wave group's partial chains go to the first, which adds them in order (all slabs are free here:
            // every wave has passed the last step's barrier and its own wait).
            static_assert(KS * L::kSlab >= RT * G * 4 * 64 * 4, "partial chains fit a slab");
            wide_barrier();
            float *red = reinterpret_cast<float *>(slabs) + (wave - ks * RT) * (G * 4 * 64) + lane;
            float *red2 = reinterpret_cast<float *>(slabs + KS * L::kSlab) + (wave - ks * RT) * (G * 4 * 64) + lane;
            if (ks == 1) {
#pragma unroll
                for (int g = 0; g < G; g++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        if constexpr (SPLIT) {
                            red2[(g * 4 + j) * 64] = acc[g][j];
                            red[(g * 4 + j) * 64] = total[g][j];
                        } else {
                            red[(g * 4 + j) * 64] = acc[g][j];
                        }
                    }
            }
            wide_barrier();
            if (ks == 1) return;
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float v = acc[g][j];
                    if constexpr (SPLIT) v = total[g][j] + v;
                    v = v + red[(g * 4 + j) * 64];
                    if constexpr (SPLIT) v = v + red2[(g * 4 + j) * 64];
                    acc[g][j] = v;
                }
        }
        const int row = tile * 16 + n - a.row_skip;
        if (tile < a.n_tiles && row >= 0 && row < a.rows) {
            float *out = (second ? a.out2 : a.out) + static_cast<int64_t>(a0 + tok0) * a.rows + row;
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int t = 16 * g + 4 * kq + j;
                    float v = acc[g][j];
                    if constexpr (SPLIT && KS == 1) v = part == 0 ? v : total[g][j] + v;
                    if (t < n_here) out[static_cast<int64_t>(t) * a.rows] = v;
                }
        }
        if constexpr (!GROUPED) return;
        wide_barrier();  // (every wave's requests have arrived: the next column may use the buffers)
    }
}

template <class F, int G, int WAVES, int KS, bool SPLIT, bool GROUPED, bool ONCE = false>
static int launch_wide(WideArgs<F> ka, int slots, hipStream_t st) {
    typedef WideLds<F, G, WAVES, KS> L;
    static_assert(L::kTotal <= 160 * 1024, "LDS of a compute unit");
    constexpr int RT = WAVES / KS;
    ka.n_tiles = (ka.rows + ka.row_skip + 15) / 16;
    ka.n_row_blocks = (ka.n_tiles + RT - 1) / RT * (ka.out2 ? 2 : 1);
    ka.n_cols = GROUPED ? 1 : (ka.n_tokens + L::NTOK - 1) / L::NTOK;
    static std::atomic<bool> raised{false};  // per instantiation: allow more than 64 KB of dynamic LDS once
    if (!raised.load(std::memory_order_acquire)) {
        CML_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_wide_kernel<F, G, WAVES, KS, SPLIT, GROUPED, ONCE>), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        raised.store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL((gemm_wide_kernel<F, G, WAVES, KS, SPLIT, GROUPED, ONCE>), dim3(wide_grid(ka.n_row_blocks, ka.n_cols), slots), dim3(64 * WAVES), L::kTotal, st, ka);
    // "<format>.mfma.wide.g<token groups>w<waves>[.ksplit2][.serial_split][.grouped][.once]"
    CML_COUNT_LAUNCH(std::string(F::kName) + ".mfma.wide.g" + std::to_string(G) + "w" + std::to_string(WAVES) + (KS == 2 ? ".ksplit2" : "") +
                     (SPLIT ? ".serial_split" : "") + (GROUPED ? ".grouped" : "") + (ONCE ? ".once" : ""));
    CML_HIP_TRY(hipGetLastError());
    return CML_OK;
}

// The shape of a launch: token groups per column, waves per workgroup, and how a K cut is walked.
struct WideShape {
    int g = 0, waves = 0, ks = 1;
};

// Estimated us of a launch (less a constant), fitted on MI355X to every shape of the kernel on cold weights (more than the last-level cache holds between
// two launches on one) of 256 to 65536 rows and 512 to 14336 values with the three K cuts: Q6_K 1669 pairs of weight and tokens (5 to 512), Q4_K 1397 (33 to
// 512).  The shape with the lowest estimate was on average 0.8 % / 0.7 % slower than the fastest (an earlier fit to few weights, some of them cached, took Q4_K
// 4.3 % off).  Q4_K has since become 1 to 4 % faster in the cells and the unpacking; with the constants as they are 276 pairs of 70 other weights, equally cold, are 1.1 % off in Q4_K (29 %
// at worst: 37336 x 1024 at 36 tokens 16.2 us, four waves on three token groups 12.6) and 279 of 70 in Q6_K, which the change left alone, 1.7 % (19 %: 42952 x 2816 at 40 38.4, 32.4).
// A step costs a fixed latency, more for two wave groups; for every wave on a SIMD the unpacking of a super-block and the cells of its token groups;
// and per token group the activation slabs that the compute unit's workgroups fetch (from three on they share what the cache holds).  Workgroups fill an XCD's 32
// compute units row block by row block (wide_block).  `rounds`: workgroups over what is resident at once, between their average and the last round at full length.
template <class F>
static float wide_cost(int64_t tiles, int groups, int n_sb, int ksplit, const WideShape &s, int lds) {
    const int rt = s.waves / s.ks;
    const int64_t blocks = (tiles + rt - 1) / rt, per_xcd = (blocks + 7) / 8 * ((groups + s.g - 1) / s.g);
    const int resident = std::min(160 * 1024 / lds, 8 / s.waves);  // (registers: two waves per SIMD)
    const float per_cu = per_xcd / 32.0f, full = per_cu / resident;
    const float rounds = full <= 1.0f ? 1.0f : 0.4f * full + 0.6f * std::ceil(full);
    const int here = per_cu > 1.0f ? resident : 1;
    const float waves = here * s.waves / 4;  // per SIMD
    const int mid = s.ks == 2 ? ksplit / 2 * n_sb / ksplit : 0, steps = std::max(mid, n_sb - mid);
    return rounds * steps * (F::kStepUs + F::kPartUs * s.ks + F::kUnpackUs * waves + s.g * (F::kCellsUs * waves + F::kSlabUs * std::min(3, s.ks * here)));
}

template <class F, int G, int WAVES, int KS>
static void wide_consider(int64_t tiles, int groups, int n_sb, int ksplit, WideShape &best, float &cost) {
    typedef WideLds<F, G, WAVES, KS> L;
    if constexpr (L::kTotal <= 160 * 1024) {
        const WideShape s{G, WAVES, KS};
        const float c = wide_cost<F>(tiles, groups, n_sb, ksplit, s, L::kTotal);
        if (c < cost) {
            cost = c;
            best = s;
        }
    }
}

template <class F, int WAVES, int KS>
static void wide_consider_g(int64_t tiles, int groups, int n_sb, int ksplit, WideShape &best, float &cost) {
    wide_consider<F, 1, WAVES, KS>(tiles, groups, n_sb, ksplit, best, cost);
    wide_consider<F, 2, WAVES, KS>(tiles, groups, n_sb, ksplit, best, cost);
    wide_consider<F, 3, WAVES, KS>(tiles, groups, n_sb, ksplit, best, cost);
    wide_consider<F, 4, WAVES, KS>(tiles, groups, n_sb, ksplit, best, cost);
    wide_consider<F, 5, WAVES, KS>(tiles, groups, n_sb, ksplit, best, cost);
    wide_consider<F, 6, WAVES, KS>(tiles, groups, n_sb, ksplit, best, cost);
    wide_consider<F, 7, WAVES, KS>(tiles, groups, n_sb, ksplit, best, cost);
    wide_consider<F, 8, WAVES, KS>(tiles, groups, n_sb, ksplit, best, cost);
}

template <class F, int G, int WAVES, int KS>
static int launch_wide_split(const WideArgs<F> &ka, hipStream_t st) {
    if constexpr (WideLds<F, G, WAVES, KS>::kTotal <= 160 * 1024) {
        const bool split = KS == 2 ? ka.ksplit > 2 : ka.ksplit > 1;
        return split ? launch_wide<F, G, WAVES, KS, true, false>(ka, 1, st) : launch_wide<F, G, WAVES, KS, false, false>(ka, 1, st);
    } else {
        return fail(CML_ERR_UNSUPPORTED, "wide matrix-core kernel: no such shape");
    }
}

template <class F, int WAVES, int KS>
static int launch_wide_g(const WideArgs<F> &ka, int g, hipStream_t st) {
    switch (g) {
        case 1: return launch_wide_split<F, 1, WAVES, KS>(ka, st);
        case 2: return launch_wide_split<F, 2, WAVES, KS>(ka, st);
        case 3: return launch_wide_split<F, 3, WAVES, KS>(ka, st);
        case 4: return launch_wide_split<F, 4, WAVES, KS>(ka, st);
        case 5: return launch_wide_split<F, 5, WAVES, KS>(ka, st);
        case 6: return launch_wide_split<F, 6, WAVES, KS>(ka, st);
        case 7: return launch_wide_split<F, 7, WAVES, KS>(ka, st);
        default: return launch_wide_split<F, 8, WAVES, KS>(ka, st);
    }
}

template <class F>
static int launch_wide_plain(const MatArgs &a, hipStream_t st) {
    const cml_weight *w = a.w;
    WideArgs<F> ka{};
    ka.w = F::weight(w);
    ka.rows = static_cast<int>(w->rows);
    ka.row_skip = w->row_skip;
    ka.n_sb = static_cast<int>(w->nb);
    ka.ksplit = F::ksplit(w->rows, w->nb);
    ka.q = a.q;
    ka.yd = a.scales;
    ka.out = a.out;
    ka.n_tokens = static_cast<int>(a.n_tokens);
    const int64_t tiles = (w->rows + w->row_skip + 15) / 16;
    const int groups = (ka.n_tokens + 15) / 16;
    WideShape s;
    float cost = 1e30f;
    const bool two = ka.ksplit == 2 || ka.ksplit == 4;  // (other cuts are closed inside the lane)
    wide_consider_g<F, 4, 1>(tiles, groups, ka.n_sb, ka.ksplit, s, cost);
    wide_consider_g<F, 8, 1>(tiles, groups, ka.n_sb, ka.ksplit, s, cost);
    if (two) {
        wide_consider_g<F, 4, 2>(tiles, groups, ka.n_sb, ka.ksplit, s, cost);
        wide_consider_g<F, 8, 2>(tiles, groups, ka.n_sb, ka.ksplit, s, cost);
    }
    // (forced shapes: tests and measurements.  Of the 31 / 32 compiled ones the estimate never takes, over 1 to 9500 tiles, 1 to 128 groups and the three cuts, Q4_K 8 groups and
    // 4 to 8 on two parts with four waves, Q6_K eight waves alone and with 1 to 4 groups on two parts: the tests' other implementations of the same cells)
    s.g = env_int("CAMELID_HIP_WIDE_GROUPS", s.g);
    s.waves = env_int("CAMELID_HIP_WIDE_WAVES", s.waves);
    s.ks = two ? env_int("CAMELID_HIP_WIDE_PARTS", s.ks) : 1;
    if (s.ks == 2) return s.waves == 4 ? launch_wide_g<F, 4, 2>(ka, s.g, st) : launch_wide_g<F, 8, 2>(ka, s.g, st);
    return s.waves == 4 ? launch_wide_g<F, 4, 1>(ka, s.g, st) : launch_wide_g<F, 8, 1>(ka, s.g, st);
}

// Expert groups: four waves up to 64 assignments (three workgroups per compute unit up to 48), eight beyond; token groups per column enough for most groups of a
// routing whose assignments fall evenly (mean and one deviation; with one and a half, three token groups where two are enough: layer of 8 experts, top-2, at 100 tokens
// 2048 / 8192 101 -> 109 us, 4096 / 14336 241 -> 247); a fuller group takes another column, groups of 16 past a group's last are skipped.
template <class F, int G, int WAVES>
static int launch_wide_grouped_split(const WideArgs<F> &ka, int slots, bool once, hipStream_t st) {
    if (once) return ka.ksplit > 1 ? launch_wide<F, G, WAVES, 1, true, true, true>(ka, slots, st) : launch_wide<F, G, WAVES, 1, false, true, true>(ka, slots, st);
    return ka.ksplit > 1 ? launch_wide<F, G, WAVES, 1, true, true>(ka, slots, st) : launch_wide<F, G, WAVES, 1, false, true>(ka, slots, st);
}

template <class F>
static int launch_wide_grouped(const MatArgs &a, hipStream_t st) {
    const cml_weight *w = a.w;
    WideArgs<F> ka{};
    ka.w = F::weight(w);
    ka.rows = static_cast<int>(a.band_rows);
    ka.n_sb = static_cast<int>(w->nb);
    ka.ksplit = F::ksplit(ka.rows, w->nb);
    ka.q = a.q;
    ka.yd = a.scales;
    ka.out = a.out;
    ka.n_tokens = static_cast<int>(a.n_tokens);
    ka.group_offsets = a.group_offsets;
    ka.group_rows = a.group_rows;
    ka.group_ids = a.group_ids;
    if (a.w2) {
        ka.w2 = F::weight(a.w2);
        ka.out2 = a.out2;
    }
    const int slots = static_cast<int>(a.group_ids ? a.max_active : a.n_groups);
    const float mean = static_cast<float>(a.n_assign_total) / std::max(1, slots);
    int g = static_cast<int>(std::ceil(std::min<float>(mean + std::sqrt(mean), static_cast<float>(ka.n_tokens)) / 16.0f));
    g = env_int("CAMELID_HIP_WIDE_GROUPS", g);
    const bool once = wide_reads_once(w);
    if (g <= 2) return launch_wide_grouped_split<F, 2, 4>(ka, slots, once, st);
    if (g <= 3) return launch_wide_grouped_split<F, 3, 4>(ka, slots, once, st);
    if (g <= 4) return launch_wide_grouped_split<F, 4, 4>(ka, slots, once, st);
    return launch_wide_grouped_split<F, 8, 8>(ka, slots, once, st);
}

}  // namespace cml
