// Q8_0 / Q4_0 x Q8_0 matmul for prefill batches and expert groups on the int8 matrix cores (gfx950).
//
// Arithmetic: cell by cell that of the matvec kernels and of gemm_b32_mfma.hip: per 32-value block, in block order,
//     isum = sum_j w_j * x_j  (exact i32),   acc = acc + ((float)isum * d_w) * d_x
// so one v_mfma_i32_16x16x32_i8 per block and 16 x 16 cells, and an f32 step per block and cell: the vector
// instructions bound this kernel (three per 64 cells and block, the fused one four cycles and the others two with two waves to take turns: 14336 x 4096 x 200 tokens
// 24 us of issue, 57 measured: in row blocks of 128 and columns of 4, 3, 3, 3 token groups a compute unit has up to 7 groups where 5.7 is the mean).  Three
// are the least: multiply, multiply, add, each rounded.  The conversion is left out: the matrix instruction
// adds onto 0x4b400000, so that its result READ AS f32 is 12582912 + isum (|isum| <= 2^19), and
//     fma(that, d_w, -12582912 * d_w)
// is isum * d_w rounded once, the product (d_w has 11 significant bits, 1.5 * 2^23 * d_w is exact).  A slab
// that holds a scale which is no finite number takes the subtraction instead (inf - inf).
//
// A wave owns one or two 16-row tiles (RT) and all tokens of its workgroup's column.  With two, an activation operand and the activation scales read from
// LDS serve both, with one a launch has more workgroups and a compute unit room for more of them: b32_wide_cost chooses.
// K is walked in slabs of 256 values.  Everything a slab needs goes from memory to LDS without passing through
// registers (gemm_wide.hpp): the activation of the workgroup's tokens and their scales (D + 1 buffers), the rows
// of every wave (D buffers: a wave holds the slab it works on in registers).  LDS is written at consecutive
// addresses, 16 bytes per lane; bank conflicts are avoided by what each lane fetches (exclusive-or of the piece with the row).
// Lane L supplies A-row t = L % 16 and B-column n = L % 16 at the k-octet L / 16 of a block and
// receives D[4 * (L / 16) + j][L % 16], j < 4.  Q4_0: octets 0, 1 are the low nibbles of the block's first and second
// eight bytes, octets 2, 3 the high ones.
// With one token group the weight costs Q4_0 more than the cells do: its words and scales are converted where they are used, in four instructions per word pair and two per
// scale where they were eight and four, and in registers enough fewer that four waves fit a SIMD (32000 x 4096 at 16 tokens 22.8 -> 20.2 us, 4096 x 14336 46 -> 39).
// Rows of no whole slabs (cols no multiple of 256) had the packed dot alone, eight tokens per pass over the weight: 4096 x 4160 at 16 / 40 / 200 tokens 31.5 -> 16.1,
// 78 -> 16.5, 394 -> 26.6 us, 14336 x 2912 at 64 161 -> 23.5.
// us per launch, gemm_b32_mfma.hip -> here: Q8_0 14336 x 4096 at 24 / 64 / 200 / 512 tokens 34.5 -> 21.2, 67 -> 24, 217 -> 58,
// 434 -> 115 (523 TOP/s); 4096 x 14336 at 64 / 512 73 -> 39, 541 -> 116; Q4_0 128256 x 3072 at 16 / 64 57.7 -> 51, 156 -> 100.
#include "gemm_wide.hpp"

#pragma clang fp contract(off)

namespace cml {

typedef int v2i_w __attribute__((ext_vector_type(2)));

struct B32WideArgs {
    const uint8_t *quants;  // plane 0, row-major
    const uint8_t *scales;  // plane 1: f16 per block, row-major
    int64_t q_stride, s_stride;
    int rows, n_slabs;
    int nb;            // blocks per row
    bool once;         // (chooses the kernel)
    int n_row_blocks, n_cols;
    int base, more;    // token groups of a column; columns that have one more
    const int8_t *q;   // [n_tokens][nb*32]
    const float *xs;   // [n_tokens][nb], 16-byte aligned (rows of whole slabs)
    float *out;        // [n_tokens][rows]
    int n_tokens;
    // Grouped call (mixture of experts), as in WideArgs: blockIdx.y -> group, its band of rows and its assignments.
    const int32_t *group_offsets;
    const int32_t *group_rows;
    const int32_t *group_ids;
};

constexpr int kB32Waves = 4;

typedef unsigned short us2_w __attribute__((ext_vector_type(2)));
typedef _Float16 h2_w __attribute__((ext_vector_type(2)));

// The eight bytes of a block that a lane holds, as the matrix instruction's operand.  Q4_0: the nibbles of its k-quarter (low ones in lanes of quarters
// 0 and 1) in the upper half of the bytes with the top bit turned over, 16 (nibble - 8): two instructions per word, four to bring nibble - 8 down.
template <int FMT>
__device__ __forceinline__ v2i_w b32_operand(v2i_w o, int kq) {
    if constexpr (FMT == CML_Q8_0) return o;
    const int up = 4 - 4 * (kq >> 1);
    return v2i_w{static_cast<int>(((static_cast<uint32_t>(o.x) << up) & 0xf0f0f0f0u) ^ 0x80808080u), static_cast<int>(((static_cast<uint32_t>(o.y) << up) & 0xf0f0f0f0u) ^ 0x80808080u)};
}
// d_w, over the 16 that a Q4_0 operand carries (both steps exact: 2^-28 is a normal f32)
template <int FMT>
__device__ __forceinline__ float b32_scale(uint32_t two, int odd) {
    const h2_w h = __builtin_bit_cast(h2_w, two);
    const float d = static_cast<float>(odd ? h.y : h.x);
    return FMT == CML_Q8_0 ? d : d * 0.0625f;
}

// LDS layout of one workgroup.
template <int FMT, int G, int RT, int D, bool RAGGED>
struct B32WideLds {
    static constexpr int NTOK = 16 * G;
    static constexpr int kRowBytes = FMT == CML_Q8_0 ? 256 : 128;
    static constexpr int kSlab = NTOK * 256;
    static constexpr int kXs = (NTOK + 31) / 32 * 1024;         // activation scales [token][8]
    static constexpr int kQuants = RT * 16 * kRowBytes;         // of a wave's rows
    static constexpr int kScales = RAGGED ? 512 : 256;          // block scales of 16 rows, [row][8] f16; RAGGED: the eight aligned words from the first on
    static constexpr int kWave = kQuants + RT * kScales;
    static constexpr int kTotal = (D + 1) * (kSlab + kXs) + D * kB32Waves * kWave;
};

// G: token groups of 16 per column.  RT: row tiles of a wave.  D: slabs requested ahead.
// GROUPED: expert groups; a workgroup walks all token columns of its group.  ONCE: the weight is requested past the caches (wide_reads_once) where one column
// reads it: of expert groups, whose sizes only the device knows, by the workgroups of those that fill one column at most.
// RAGGED: rows of no whole slabs.  Their last slab is short: requests past the row repeat its last piece, the blocks it does not have take no f32 step;
// scale rows may start at any even address, activation scales come a word per lane.
template <int FMT, int G, int RT, int D, bool GROUPED, bool ONCE, bool RAGGED>
__global__ __launch_bounds__(64 * kB32Waves, FMT == CML_Q4_0 && G == 1 ? 5 - RT - RAGGED : 2) void gemm_b32_wide_kernel(B32WideArgs a) {
    typedef B32WideLds<FMT, G, RT, D, RAGGED> L;
    constexpr int NTOK = L::NTOK, WAVES = kB32Waves;
    constexpr int kThreads = 64 * WAVES;
    constexpr bool kLate = FMT == CML_Q4_0 && G == 1;  // a slab's weight is used once: it is unpacked where it is used
    static_assert(kThreads == 256, "a pass of the workgroup fetches a token group");
    static_assert(!GROUPED || D == 1, "waves of a grouped call may have fewer requests in flight");
    extern __shared__ uint4 smem[];
    uint8_t *slabs = reinterpret_cast<uint8_t *>(smem);  // [D + 1][NTOK][256]
    constexpr int kXsAt = (D + 1) * L::kSlab, kWAt = kXsAt + (D + 1) * L::kXs;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int n = lane & 15, kq = lane >> 4;
    int row_block, col;
    if (!wide_block(blockIdx.x, a.n_row_blocks, a.n_cols, row_block, col)) return;
    const int64_t band = GROUPED ? (a.group_ids ? a.group_ids[blockIdx.y] : static_cast<int>(blockIdx.y)) : 0;
    if (band < 0) return;  // a slot past the groups in use
    const int a0 = GROUPED ? a.group_offsets[band] : 0;
    const int n_assign = GROUPED ? a.group_offsets[band + 1] - a0 : a.n_tokens;
    // The walk over K of one column of NG token groups.
    auto walk = [&](int tok0, int n_here, auto groups, auto once) __attribute__((always_inline)) {
        constexpr int NG = decltype(groups)::value;
        auto act_row = [&](int t) __attribute__((always_inline)) -> uint32_t {  // (tokens past the end repeat the last one)
            const int j = min(t, n_here - 1);
            return static_cast<uint32_t>(GROUPED ? (a.group_rows ? a.group_rows[a0 + tok0 + j] : a0 + tok0 + j) : j);
        };
        const int n_slabs = a.n_slabs;
        const int row0 = (row_block * WAVES + wave) * (16 * RT);

        const uint32_t lds0 = lds_address(smem);
        // Activation: thread tid fetches slot tid % 16 of tokens tid / 16 + 16 * k.
        const int t16 = tid >> 4, piece = (tid & 15) ^ (t16 & 15);
        const uint32_t row_bytes = RAGGED ? a.nb * 32u : n_slabs * 256u;
        const int8_t *q_base = a.q + (GROUPED ? 0 : static_cast<int64_t>(tok0) * row_bytes);
        uint32_t src[NG];
#pragma unroll
        for (int k = 0; k < NG; k++) src[k] = act_row(t16 + 16 * k) * row_bytes + piece * 16;
        // Scales: lane pairs of the first waves, token 32 * wave + lane / 2; RAGGED: eight tokens per request, a block per lane.
        const bool xs_wave = wave < L::kXs / 1024;
        const float *xs_base = a.xs + (GROUPED ? 0 : static_cast<int64_t>(tok0) * (RAGGED ? a.nb : n_slabs * 8));
        const uint32_t xs_src = RAGGED ? 0 : act_row(32 * wave + (lane >> 1)) * (n_slabs * 32u) + (lane & 1) * 16;
        constexpr int kXsReqs = RAGGED ? (NG + 1) / 2 : 0;
        uint32_t xs_row[RAGGED ? kXsReqs : 1];
#pragma unroll
        for (int i = 0; i < kXsReqs; i++) xs_row[i] = act_row(8 * wave + 32 * i + (lane >> 3)) * (a.nb * 4u);
        auto fetch = [&](int slab, int buf) __attribute__((always_inline)) {
            slab = min(slab, n_slabs - 1);
            uint32_t cut = 0;  // what a lane's piece lies past the row
            if constexpr (RAGGED) {
                const int left = a.nb - 8 * slab;
                cut = max(piece - 2 * left + 1, 0) * 16;
                const uint32_t block = min(lane & 7, left - 1) * 4;
#pragma unroll
                for (int i = 0; i < kXsReqs; i++)
                    if (wave + 4 * i < 2 * NG)  // (the address in a scalar register, which the compiler does not see to by itself)
                        wide_dma4(__builtin_amdgcn_readfirstlane(lds0 + kXsAt + buf * L::kXs + (wave + 4 * i) * 256), xs_base + slab * 8, xs_row[i] + block);
            } else if (xs_wave) {
                wide_dma16(lds0 + kXsAt + buf * L::kXs + wave * 1024, xs_base + slab * 8, xs_src);
            }
#pragma unroll
            for (int k = 0; k < NG; k++)
                if (!GROUPED || 4 * wave + 16 * k < n_here)  // (what no token owns stays what it was: cells of its own, never stored)
                    wide_dma16(lds0 + buf * L::kSlab + k * (16 * kThreads) + wave * 1024, q_base + slab * 256, src[k] - cut);
        };
        // Weights: rows past the end repeat the last one.
        const int first = min(row0, a.rows - 1), last = a.rows - 1 - first;  // (of this wave's rows)
        const uint8_t *wq = a.quants + (band * a.rows + first) * a.q_stride;
        const uint8_t *wd = a.scales + (band * a.rows + first) * a.s_stride;
        constexpr int kRowsReq = 1024 / L::kRowBytes, kReqs = L::kQuants / 1024;
        const uint32_t w_lds = lds0 + kWAt + wave * L::kWave;  // + slot * WAVES * kWave
        auto w_row = [&](int i) __attribute__((always_inline)) { return kRowsReq * i + lane / (64 / kRowsReq); };
        auto w_piece = [&](int i) __attribute__((always_inline)) {
            const int slot = lane % (64 / kRowsReq), r = w_row(i);
            return FMT == CML_Q8_0 ? slot ^ (r & 15) : slot ^ ((r >> 1) & 7);
        };
        uint32_t w_src[kReqs];
#pragma unroll
        for (int i = 0; i < kReqs; i++) w_src[i] = static_cast<uint32_t>(min(w_row(i), last)) * static_cast<uint32_t>(a.q_stride) + w_piece(i) * 16;
        // Scales: four lanes per row; RAGGED: eight, from the aligned word that holds the slab's first scale (wd need not be one) up to the row's last word.
        const uint32_t wd_off = RAGGED ? static_cast<uint32_t>(reinterpret_cast<uintptr_t>(wd) & 3) : 0;
        constexpr int kDReqs = L::kScales / 256 * RT;
        uint32_t d_src[kDReqs], d_end[RAGGED ? kDReqs : 1];
#pragma unroll
        for (int r = 0; r < kDReqs; r++) {
            if constexpr (RAGGED) {
                const uint32_t row_at = wd_off + static_cast<uint32_t>(min(8 * r + (lane >> 3), last)) * static_cast<uint32_t>(a.s_stride);
                d_src[r] = (row_at & ~3u) + (lane & 7) * 4;
                d_end[r] = (row_at + 2 * a.nb - 1) & ~3u;
            } else {
                d_src[r] = static_cast<uint32_t>(min(16 * r + (lane >> 2), last)) * static_cast<uint32_t>(a.s_stride) + (lane & 3) * 4;
            }
        }
        auto fetch_w = [&](int slab, int slot) __attribute__((always_inline)) {
            slab = min(slab, n_slabs - 1);
            const uint32_t to = w_lds + slot * (WAVES * L::kWave);
            const int pieces = RAGGED ? (FMT == CML_Q8_0 ? 2 : 1) * (a.nb - 8 * slab) : 0;  // of the row from this slab on
#pragma unroll
            for (int i = 0; i < kReqs; i++) {
                uint32_t from = w_src[i];
                if constexpr (RAGGED) from -= max(w_piece(i) - pieces + 1, 0) * 16;
                wide_dma16_hint<decltype(once)::value>(to + i * 1024, wq + slab * L::kRowBytes, from);
            }
#pragma unroll
            for (int r = 0; r < kDReqs; r++) {
                if constexpr (RAGGED) wide_dma4(to + L::kQuants + r * 256, wd - wd_off, min(d_src[r] + slab * 16, d_end[r]));
                else wide_dma4(to + L::kQuants + r * 256, wd + slab * 16, d_src[r]);
            }
        };
        constexpr int kAhead = (D - 1) * (NG + kReqs + kDReqs);  // requests that may be outstanding at the end of a step (some waves have more)

        // Operands of a slab: the lane's octet of the eight blocks of either tile's row, the blocks' scales.  With one token group they are
        // used once and stay as they were read until then (28 registers fewer per tile: a third or fourth wave on a SIMD).
        v2i_w bw[RT][8];
        uint32_t dh[RT][4];                                             // scales of two blocks each, as read
        float dw[kLate ? 1 : RT][kLate ? 1 : 8], md[kLate ? 1 : RT][kLate ? 1 : 8];  // d_w; -12582912 * d_w
        bool finite = true;
        auto read_w = [&](int slot) __attribute__((always_inline)) {
            const uint8_t *w_mine = slabs + kWAt + wave * L::kWave + slot * (WAVES * L::kWave);
            us2_w high = {0, 0};
#pragma unroll
            for (int r = 0; r < RT; r++) {
                const int row = 16 * r + n;
                const uint8_t *scales = w_mine + L::kQuants + row * (L::kScales / 16);
                const uint4 d = *reinterpret_cast<const uint4 *>(scales);
                dh[r][0] = d.x;
                dh[r][1] = d.y;
                dh[r][2] = d.z;
                dh[r][3] = d.w;
                if constexpr (RAGGED) {
                    // (a row past the end repeats the last one, whose parity counts)
                    const uint32_t up = ((wd_off + static_cast<uint32_t>(min(row, last)) * static_cast<uint32_t>(a.s_stride)) & 2) * 8;  // 16: the first scale is the upper half of its word
                    const uint32_t fifth = reinterpret_cast<const uint32_t *>(scales)[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) dh[r][i] = __builtin_amdgcn_alignbit(i < 3 ? dh[r][i + 1] : fifth, dh[r][i], up);
                }
#pragma unroll
                for (int b = 0; b < 8; b++) {
                    if constexpr (FMT == CML_Q8_0) bw[r][b] = *reinterpret_cast<const v2i_w *>(w_mine + row * 256 + (((2 * b + (kq >> 1)) ^ n) << 4) + (kq & 1) * 8);
                    else bw[r][b] = *reinterpret_cast<const v2i_w *>(w_mine + row * 128 + ((b ^ ((n >> 1) & 7)) << 4) + (kq & 1) * 8);
                    if constexpr (!kLate) {
                        bw[r][b] = b32_operand<FMT>(bw[r][b], kq);
                        dw[r][b] = b32_scale<FMT>(dh[r][b >> 1], b & 1);
                        md[r][b] = -12582912.0f * dw[r][b];
                        if (b & 1) high = __builtin_elementwise_max(high, __builtin_bit_cast(us2_w, dh[r][b >> 1] & 0x7c007c00u));
                    }
                }
            }
            if constexpr (!kLate) {
                finite = __builtin_amdgcn_ballot_w64(max(high.x, high.y) == 0x7c00) == 0;
                __builtin_amdgcn_sched_barrier(0);  // (in front of the workgroup barrier: behind it the check is 0.04 us of every slab)
            }
        };

        // A operand of block b: octet kq of token n; the blocks' scales of tokens 4 kq .. + 3
        uint32_t a_addr[8];
#pragma unroll
        for (int b = 0; b < 8; b++) a_addr[b] = n * 256 + (((2 * b + (kq >> 1)) ^ n) << 4) + (kq & 1) * 8;

#pragma unroll
        for (int i = 0; i < D; i++) {
            fetch(i, i);
            fetch_w(i, i);
        }
        wide_wait<kAhead>();
        read_w(0);
        wide_barrier();

        float acc[RT][NG][4];
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int g = 0; g < NG; g++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[r][g][j] = 0.0f;

        const v4i_w magic = {0x4b400000, 0x4b400000, 0x4b400000, 0x4b400000};

        auto step = [&](const uint8_t *slab, const float *xs, int blocks, auto fin, auto tail) __attribute__((always_inline)) {
            // Software pipeline over units of two blocks of a token group: while the matrix cores work on unit i + 1, the
            // f32 steps of unit i run and the operands of unit i + 2 are read.
            constexpr int kUnits = NG * 4;
            long av[3][2];
            float4 xv[2][4];  // scales of four blocks, of the lane's four tokens
            v4i_w d[2][RT][2];
            auto read_a = [&](int i) __attribute__((always_inline)) {
                const int g = i >> 2, u = i & 3;
#pragma unroll
                for (int e = 0; e < 2; e++) av[i % 3][e] = *reinterpret_cast<const long *>(slab + a_addr[2 * u + e] + g * 4096);
            };
            auto read_x = [&](int i) __attribute__((always_inline)) {  // of units i and i + 1
                const int g = i >> 2, h = (i >> 1) & 1;
#pragma unroll
                for (int j = 0; j < 4; j++) xv[h][j] = *reinterpret_cast<const float4 *>(xs + (16 * g + 4 * kq + j) * 8 + 4 * h);
            };
            auto contract = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 2; e++)
#pragma unroll
                    for (int r = 0; r < RT; r++) {
                        const v2i_w w = kLate ? b32_operand<FMT>(bw[r][2 * (i & 3) + e], kq) : bw[r][2 * (i & 3) + e];
                        d[i & 1][r][e] = __builtin_amdgcn_mfma_i32_16x16x32_i8(av[i % 3][e], __builtin_bit_cast(long, w), magic, 0, 0, 0);
                    }
            };
            auto chain = [&](int i) __attribute__((always_inline)) {
                const int g = i >> 2, u = i & 3, h = u >> 1;
#pragma unroll
                for (int e = 0; e < 2; e++) {
                    const int b = 2 * u + e, k = 2 * (u & 1) + e;
                    if (decltype(tail)::value && b >= blocks) continue;
                    float late[RT];
#pragma unroll
                    for (int r = 0; r < RT; r++) late[r] = kLate ? b32_scale<FMT>(dh[r][b >> 1], b & 1) : 0.0f;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float x = k == 0 ? xv[h][j].x : k == 1 ? xv[h][j].y : k == 2 ? xv[h][j].z : xv[h][j].w;
#pragma unroll
                        for (int r = 0; r < RT; r++) {
                            const float f = __builtin_bit_cast(float, static_cast<int>(d[i & 1][r][e][j]));
                            const float d_w = kLate ? late[r] : dw[kLate ? 0 : r][kLate ? 0 : b];
                            const float p = !kLate && decltype(fin)::value ? __builtin_fmaf(f, d_w, md[kLate ? 0 : r][kLate ? 0 : b]) : (f - 12582912.0f) * d_w;
                            acc[r][g][j] = acc[r][g][j] + p * x;
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < RT; r++)
#pragma unroll
                    for (int j = 0; j < 4; j++) asm volatile("" : "+v"(acc[r][g][j]));  // (keeps the compiler from sinking the chains to the store)
            };
            read_a(0);
            read_x(0);
            read_a(1);
            contract(0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < kUnits; i++) {
                if (i + 2 < kUnits) {
                    read_a(i + 2);
                    if ((i & 1) == 0) read_x(i + 2);
                }
                if (i + 1 < kUnits) contract(i + 1);
                chain(i);
                __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);
#pragma unroll
                for (int m = 0; m < 2 * RT; m++) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, kLate ? 22 : 12, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };

        int buf = 0, slot = 0;  // of slab s: s % (D + 1), s % D
        for (int s = 0; s < n_slabs; s++) {
            fetch(s + D, buf == 0 ? D : buf - 1);  // (past the end the last slab again; the buffer of slab s - 1)
            fetch_w(s + D, slot);                  // (slab s was read into registers before the barrier)
            __builtin_amdgcn_sched_barrier(0);
            const uint8_t *slab = slabs + buf * L::kSlab;
            const float *xs = reinterpret_cast<const float *>(slabs + kXsAt + buf * L::kXs);
            if (RAGGED && s == n_slabs - 1) step(slab, xs, a.nb - 8 * s, std::false_type{}, std::integral_constant<bool, RAGGED>{});
            else if (kLate || !finite) step(slab, xs, 8, std::false_type{}, std::false_type{});
            else step(slab, xs, 8, std::true_type{}, std::false_type{});
            wide_wait<kAhead>();
            buf = buf == D ? 0 : buf + 1;
            slot = slot == D - 1 ? 0 : slot + 1;
            read_w(slot);
            wide_barrier();
        }
        wide_wait<0>();  // (nothing may still be on its way into LDS that is given back)

#pragma unroll
        for (int r = 0; r < RT; r++) {
            const int row = row0 + 16 * r + n;
            if (row < a.rows) {
                float *out = a.out + static_cast<int64_t>(a0 + tok0) * a.rows + row;
#pragma unroll
                for (int g = 0; g < NG; g++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int t = 16 * g + 4 * kq + j;
                        if (t < n_here) out[static_cast<int64_t>(t) * a.rows] = acc[r][g][j];
                    }
            }
        }
    };
    if constexpr (GROUPED) {
        if constexpr (ONCE) {
            if (n_assign <= NTOK) {
                if (n_assign > 0) walk(0, n_assign, std::integral_constant<int, G>{}, std::true_type{});
                return;
            }
        }
        for (int tok0 = 0; tok0 < n_assign; tok0 += NTOK) {
            walk(tok0, min(NTOK, n_assign - tok0), std::integral_constant<int, G>{}, std::false_type{});
            wide_barrier();  // (every wave's requests have arrived: the next column may use the buffers)
        }
    } else if constexpr (G == 1) {
        walk(col * NTOK, min(NTOK, n_assign - col * NTOK), std::integral_constant<int, 1>{}, std::integral_constant<bool, ONCE>{});
    } else {
        // The columns' token groups differ by one at most: those of 13 groups in columns of up to four are 4, 3, 3, 3.  Where they do differ, every other
        // 32 workgroups of an XCD take the columns one further on: the two workgroups of a compute unit (it gets the 32nd after its first) are not both the
        // larger ones.  14336 x 4096 at 200 tokens 63.3 -> 60.6 us (Q8_0), 61.6 -> 58.4 (Q4_0) against a last column padded to four.
        const int turn = col + (a.more == 0 ? 0 : (row_block >> 3) * a.n_cols >> 5 & 1), c = turn == a.n_cols ? 0 : turn;
        const int first = 16 * (c * a.base + min(c, a.more)), here = a.base + (c < a.more ? 1 : 0);
        const int n_here = min(16 * here, n_assign - first);
        if (here == G) walk(first, n_here, std::integral_constant<int, G>{}, std::false_type{});
        else walk(first, n_here, std::integral_constant<int, G - 1>{}, std::false_type{});
    }
}

template <int FMT, int G, int RT, int D, bool GROUPED, bool ONCE, bool RAGGED>
static int launch_b32_wide_as(const B32WideArgs &ka, int slots, hipStream_t st) {
    typedef B32WideLds<FMT, G, RT, D, RAGGED> L;
    auto *kernel = &gemm_b32_wide_kernel<FMT, G, RT, D, GROUPED, ONCE, RAGGED>;
    static std::atomic<bool> raised{false};  // per instantiation: allow more than 64 KB of dynamic LDS once
    if (!raised.load(std::memory_order_acquire)) {
        CML_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        raised.store(true, std::memory_order_release);
    }
    hipLaunchKernelGGL(kernel, dim3(wide_grid(ka.n_row_blocks, ka.n_cols), slots), dim3(64 * kB32Waves), L::kTotal, st, ka);
    // "<format>.mfma.wide.g<token groups>r<row tiles of a wave>d<slabs ahead>[.ragged][.grouped][.once]"
    CML_COUNT_LAUNCH(std::string(FMT == CML_Q8_0 ? "q8_0" : "q4_0") + ".mfma.wide.g" + std::to_string(G) + "r" + std::to_string(RT) + "d" + std::to_string(D) + (RAGGED ? ".ragged" : "") + (GROUPED ? ".grouped" : "") + (ONCE ? ".once" : ""));
    CML_HIP_TRY(hipGetLastError());
    return CML_OK;
}

// Past the caches (wide_reads_once): weights of expert groups, weights of a plain call of up to 16 tokens (128256 x 3072 at 16 tokens in Q8_0 85.3 -> 79.0 us; a
// single wider column gains half of that and no kernel of its own).  Not rows of no whole slabs whose 128-byte lines hold a piece of the next row too, which the hint has
// fetched twice: any in Q4_0, in Q8_0 those of other than a multiple of four blocks (plain / so, weights that no cache holds, 8 tokens: Q8_0 32000 x 4128 42.3 / 45.2, 100000 x 2912
// 82.5 / 86.4; Q4_0 128256 x 3104 68.5 / 77.9, 65536 x 4128 59.6 / 66.6; 128 experts 2816 / 704 at 64 tokens, gate and up by the hint, down both ways: 131.0 / 136.4; but Q8_0
// 46552 x 8576 85.4 / 80.9, 84064 x 3712 71.4 / 68.0; 128 experts 1920 / 1152, Q8_0, at 64 tokens 181 / 171).
template <int FMT, int G, int RT, int D, bool GROUPED = false>
static int launch_b32_wide(B32WideArgs ka, int slots, hipStream_t st) {
    constexpr int kRows = kB32Waves * 16 * RT;
    ka.n_row_blocks = (ka.rows + kRows - 1) / kRows;
    ka.n_cols = GROUPED ? 1 : (ka.n_tokens + 16 * G - 1) / (16 * G);
    const int groups = (ka.n_tokens + 15) / 16;
    ka.base = groups / ka.n_cols;
    ka.more = groups % ka.n_cols;
    if (ka.nb % 8 != 0) {
        if constexpr (G == 4 && RT == 2) return fail(CML_ERR_UNSUPPORTED, "wide matrix-core kernel: no such shape");  // (no registers left for the ragged form)
        if constexpr (FMT == CML_Q8_0 && (GROUPED || G == 1))
            if (ka.once && ka.n_cols == 1 && ka.nb % 4 == 0) return launch_b32_wide_as<FMT, G, RT, D, GROUPED, true, true>(ka, slots, st);
        if constexpr (G < 4 || RT < 2) return launch_b32_wide_as<FMT, G, RT, D, GROUPED, false, true>(ka, slots, st);
    }
    if constexpr (GROUPED || G == 1)
        if (ka.once && ka.n_cols == 1) return launch_b32_wide_as<FMT, G, RT, D, GROUPED, true, false>(ka, slots, st);
    return launch_b32_wide_as<FMT, G, RT, D, GROUPED, false, false>(ka, slots, st);
}

struct B32WideShape {
    int g = 0, rt = 0, d = 0;
};

// Workgroups that a compute unit holds by registers.
static int b32_wide_resident(int fmt, bool ragged, const B32WideShape &s) {
    if (s.rt == 2) return fmt == CML_Q4_0 && s.g == 1 && !ragged ? 3 : 2;
    if (s.g == 1) return fmt == CML_Q4_0 && !ragged ? 4 : 3;
    return s.g == 2 || (s.g == 3 && !ragged) ? 3 : 2;
}

// Estimated us of a launch (less a constant), fitted on MI355X to 2640 pairs of weight and tokens in every shape on cold weights (more than the last-level cache
// holds between two launches on one): both formats, rows of whole slabs (152 weights) and of no whole ones (84), 512 to 152064 rows, 512 to 14336 values, 5 to 400 tokens.
// A slab costs a fixed latency and, for every wave on a SIMD and row tile, 0.19 us (Q4_0 0.16, 0.14 where it is unpacked at its one use) and 0.18 (0.16) per token group; a wave
// alone on its SIMD stalls where others overlap (1.9, not 1, times that).  A second slab ahead shortens the latency of workgroups that have a compute unit of their own (8 tokens,
// one slab ahead / two: 4096 x 4096 Q8_0 17.8 / 13.5 us; 14336 x 5120 27.4 / 19.2) for a longer start, on rows of no whole slabs nearly twice as long (736 x 704 at 200 tokens
// 5.0 / 6.5).  Workgroups fill an XCD's 32 compute units row block by row block (wide_block), and the compute unit that holds the most of them is the last.  The shape with the
// lowest estimate is on average 0.7 % slower than the fastest, 17 % at worst; on 1000 other weights (5200 pairs) 0.6 % and 16 % (the estimate before, which took the residence of
// whole slabs for rows of none, 1.4 % and 49 %; calls moved either way: Q4_0 105120 x 608 at 8 tokens 16.3 -> 18.3, 139360 x 1728 at 8 50.1 -> 39.8).
static float b32_wide_cost(int fmt, bool ragged, int rows, int groups, int n_slabs, const B32WideShape &s) {
    const int64_t blocks = (rows + s.rt * 64 - 1) / (s.rt * 64), per_xcd = (blocks + 7) / 8 * ((groups + s.g - 1) / s.g);
    const int resident = b32_wide_resident(fmt, ragged, s);
    const float per_cu = per_xcd / 32.0f, full = per_cu / resident;
    const bool shared = per_cu > 1.0f;
    const float rounds = full <= 1.0f ? 1.0f : 0.35f * full + 0.65f * std::ceil(full);
    const float base = shared ? 0.32f : s.d == 1 ? 0.56f : 0.26f;
    const float waves = shared ? std::min<float>(resident, std::ceil(per_cu)) : 1.9f;
    const float weight = fmt == CML_Q8_0 ? 0.19f : s.g == 1 ? 0.14f : 0.16f, cells = fmt == CML_Q8_0 ? 0.18f : 0.16f;
    return rounds * (n_slabs * (base + waves * s.rt * (weight + cells * s.g)) + (s.d == 1 ? 0.0f : ragged ? 0.9f : 0.5f));
}

template <int FMT, int G, int RT, int D>
static int b32_wide_visit(const B32WideArgs &ka, B32WideShape &best, float &cost, const B32WideShape *launch, hipStream_t st) {
    typedef B32WideLds<FMT, G, RT, D, true> L;
    static_assert(2 * L::kTotal <= 160 * 1024, "two workgroups per compute unit");
    if (launch) return launch->g == G && launch->rt == RT && launch->d == D ? launch_b32_wide<FMT, G, RT, D>(ka, 1, st) : -1;
    const B32WideShape s{G, RT, D};
    const int groups = (ka.n_tokens + 15) / 16;
    if (G == 4 && RT == 2 && ka.nb % 8 != 0) return -1;
    if (G > 1 && (groups + G - 1) / G == (groups + G - 2) / std::max(1, G - 1)) return -1;  // (as few columns have room with a group less)
    const float c = b32_wide_cost(FMT, ka.nb % 8 != 0, ka.rows, groups, ka.n_slabs, s);
    if (c < cost) {
        cost = c;
        best = s;
    }
    return -1;
}

// Every shape in turn: considers it (launch null) or, if it is the wanted one, launches it.
template <int FMT, int I = 0>
static int b32_wide_each(const B32WideArgs &ka, B32WideShape &best, float &cost, const B32WideShape *launch, hipStream_t st) {
    if constexpr (I < 9) {
        const int rc = b32_wide_visit<FMT, I == 8 ? 1 : I % 4 + 1, I == 8 ? 1 : I / 4 + 1, I == 8 ? 2 : 1>(ka, best, cost, launch, st);
        return rc != -1 ? rc : b32_wide_each<FMT, I + 1>(ka, best, cost, launch, st);
    }
    return launch ? fail(CML_ERR_UNSUPPORTED, "wide matrix-core kernel: no such shape") : CML_OK;
}

template <int FMT>
static int launch_b32_wide_fmt(const B32WideArgs &ka, hipStream_t st) {
    B32WideShape s;
    float cost = 1e30f;
    b32_wide_each<FMT>(ka, s, cost, nullptr, st);
    // (forced shapes: tests and measurements)
    s.g = env_int("CAMELID_HIP_WIDE_GROUPS", s.g);
    s.rt = env_int("CAMELID_HIP_WIDE_TILES", s.rt);
    s.d = env_int("CAMELID_HIP_WIDE_AHEAD", s.d);
    return b32_wide_each<FMT>(ka, s, cost, &s, st);
}

// Expert groups: columns of 16 assignments, of 32 from 12 on average (a second column of 16 reads the weight again: 32 experts, top-8, 2816 / 1408 at
// 64 tokens Q8_0 203 us with columns of 16, 185 so; at 24 tokens 117 / 122), one row tile per wave (two: 118 / 126).
template <int FMT>
static int launch_b32_wide_grouped(const B32WideArgs &ka, const MatArgs &a, hipStream_t st) {
    const int slots = static_cast<int>(a.group_ids ? a.max_active : a.n_groups);
    const int g = env_int("CAMELID_HIP_WIDE_GROUPS", a.n_assign_total >= 12 * static_cast<int64_t>(slots) ? 2 : 1);
    return g == 1 ? launch_b32_wide<FMT, 1, 1, 1, true>(ka, slots, st) : launch_b32_wide<FMT, 2, 1, 1, true>(ka, slots, st);
}

// Rows of no whole slabs (up to a slab the packed dot serves them).  The packed dot stages a row, 40 bytes per block, in 64 KB of LDS and refuses
// longer ones: they stay refused in batches too, there is no single-token result that a batch of them could equal.
bool b32_wide_ragged(const cml_weight *w) {
    return (w->fmt == CML_Q8_0 || w->fmt == CML_Q4_0) && w->nb > 8 && w->nb % 8 != 0 && w->nb <= 64 * 1024 / 40;
}

// Whether a batch on such rows is ahead here of the packed dot, which makes one pass over the weight for 4 or 8 tokens, two or three for 3 and 5 to 7.  Time here over there at
// 3 / 4 / 5 / 8 tokens on 560 weights, more than 600 MB of others between two launches on one (1500 pairs): from 768 row tiles 0.53 - 0.91 / 0.64 - 1.27 (from 1500 tiles
// 0.64 - 1.17, 0.86 on average) / 0.42 - 0.76 / 0.32 - 0.91; from 257 tiles at 5 / 8 on rows of more than 31 blocks Q8_0 0.59 - 1.02 / 0.51 - 0.97, Q4_0 0.67 - 0.87 / 0.56 - 0.81, but up to
// 512 tiles on rows of five slabs and more 0.81 - 1.15 / 0.62 - 1.00; up to 256 tiles at 5 / 7 / 8 / 9 on rows of four slabs and a part 0.82 - 0.87 / 0.6 / 0.89 - 0.93 / 0.7, of
// longer ones 0.87 - 1.43 / 0.63 - 0.96 / 0.86 - 1.21 / 0.73 - 0.88.  Rows of up to 31 blocks at 8 up to 256 tiles 1.08 - 1.32, up to 512 0.99 - 1.14; of 24 to 31, two nearly full
// steps of the packed dot's 16 lanes, at 5 up to 256 tiles 0.97 - 1.03, of fewer 0.86 - 0.97.
bool b32_wide_ragged_pays(const cml_weight *w, int64_t n) {
    const int forced = env_int("CAMELID_HIP_B32_MFMA_MIN_TOKENS", 0);
    if (!b32_wide_ragged(w) || env_int("CAMELID_HIP_MFMA_WIDE", 1) == 0) return false;
    if (forced > 0) return n >= forced;
    const int64_t tiles = (w->rows + 15) / 16, slabs = w->nb / 8;
    if (n == 3) return tiles >= 768;
    if (n == 4) return tiles >= 1500;
    if (n >= 9 || n < 3) return n >= 9;
    if (n == 8 && slabs <= 3 && tiles <= 512) return false;
    if (n == 5 && slabs == 3 && tiles <= 256) return false;
    if (tiles <= 256) return slabs <= 4;
    return n > 5 || w->fmt == CML_Q8_0 || tiles > 512 || slabs <= 4;
}

// Whether the offsets of a grouped call's activation rows fit 32 bits and its weight and scales can be read 16 bytes at a time.
bool gemm_b32_wide_serves_groups(const MatArgs &a) {
    return (b32_wide_ragged(a.w) || (b32_mfma_usable(a.w) && reinterpret_cast<uintptr_t>(a.scales) % 16 == 0)) &&
           std::max(a.n_assign_total, a.n_tokens) * a.w->nb * 32 < (int64_t{1} << 32);
}

// On a weight that b32_mfma_usable accepts, activation scales 16-byte aligned, or one of b32_wide_ragged; grouped: gemm_b32_wide_serves_groups.
int launch_gemm_b32_wide(const MatArgs &a, hipStream_t st) {
    const cml_weight *w = a.w;
    B32WideArgs ka{};
    ka.quants = w->planes.p[0];
    ka.q_stride = w->planes.row_stride[0];
    ka.scales = w->planes.p[1];
    ka.s_stride = w->planes.row_stride[1];
    ka.rows = static_cast<int>(a.group_offsets ? a.band_rows : w->rows);
    ka.n_slabs = static_cast<int>((w->nb + 7) / 8);
    ka.nb = static_cast<int>(w->nb);
    ka.once = wide_reads_once(w);
    ka.q = a.q;
    ka.xs = a.scales;
    ka.out = a.out;
    ka.n_tokens = static_cast<int>(a.n_tokens);
    ka.group_offsets = a.group_offsets;
    ka.group_rows = a.group_rows;
    ka.group_ids = a.group_ids;
    if (a.group_offsets) return w->fmt == CML_Q8_0 ? launch_b32_wide_grouped<CML_Q8_0>(ka, a, st) : launch_b32_wide_grouped<CML_Q4_0>(ka, a, st);
    return w->fmt == CML_Q8_0 ? launch_b32_wide_fmt<CML_Q8_0>(ka, st) : launch_b32_wide_fmt<CML_Q4_0>(ka, st);
}

}  // namespace cml
