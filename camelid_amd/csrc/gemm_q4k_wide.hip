// Q4_K x Q8_K on the wide matrix-core kernel (gemm_wide.hpp): batches of more than 32 tokens, but for small weights whose
// K is cut, and expert groups that hold more than a few assignments each (launch_gemm_q4k_mfma holds the lines).
//
// The integers are those of gemm_q4k_mfma.hip: the 6-bit scale of a sub-block as two 3-bit digits inside the int8 weight
// operand (S = lo + 8 hi, two contractions over the whole super-block), the mins against the sums of the
// activation's 16-value runs in one f16 instruction.  There the 16 operand words of a super-block are formed again for every 64
// tokens and the activation passes through registers on its way to LDS; here once for up to 128.
// Bound: matrix and vector instructions, which add up to nine tenths of the busy cycles, and LDS reads, a few cycles of the matrix unit each: a super-block and 16 x 16 cells take nine and a half matrix instructions, 16 vector ones and 4.6 KB of LDS.  The products of
// the scales, eight vector instructions before, come from the matrix unit (chain below).
// us per launch: 14336 x 4096 at 64 / 200 / 512 tokens, narrow kernel -> this one -> with the products of the scales from the matrix unit and fewer steps to unpack them (the last two with
// other weights between two launches on one) 19.3 -> 20.1 -> 19.4, 54 -> 38.8 -> 37.8, 98 -> 80.0 -> 77.3 (778 TOP/s); 4096 x 14336 at 200 / 512, narrow -> this one on a weight that the caches hold
// 88 -> 49, 185 -> 82; a layer of 8 experts of 4096 / 14336, top-2, at 48 / 128 tokens 217 -> 190, 340 -> 256.
#include "gemm_wide.hpp"

#pragma clang fp contract(off)

namespace cml {

int q4k_ksplit_for(int64_t rows, int64_t n_sb);  // gemv_q4k.hip: the matvec kernel's K-split policy

struct Q4KWide {
    static constexpr const char *kName = "q4k";
    static constexpr int kTileBytes = 2304, kFetches = 3;  // LDS bytes of a wave's super-block (pieces a | pieces b | headers), requests for it
    static constexpr float kStepUs = 0.25f, kPartUs = 0.10f, kUnpackUs = 0.12f, kCellsUs = 0.06f, kSlabUs = 0.09f;  // (wide_cost)
    static constexpr bool kRunSums = true;
    struct Weight {
        const uint8_t *w;  // tiled layout [super-block][tile][2304 B]: 16 headers, then pieces a and b as [16 rows][4 chunks][16 B]
        int64_t sb_stride;
    };
    static Weight weight(const cml_weight *w) { return Weight{w->planes.p[0], w->planes.row_stride[0]}; }
    static int ksplit(int64_t rows, int64_t n_sb) { return q4k_ksplit_for(rows, n_sb); }
    struct Raw {
        uint4 hdr, piece[2];
    };
    const uint8_t *base;  // the tile's entry of super-block 0 (wave-uniform)
    int64_t sb_stride;
    uint32_t piece_src, lane4;
    int kq, hdr_at, piece_at[2];
    struct Operands {
        v4i_w lo[4], hi[4];  // the values times the two digits of their sub-block's scale
        v4h_w mins;
        float scale;         // d in the lanes of even k-quarters, -dmin in the others
        float d, dmin;
    };

    // LDS: pieces a and b of 16 rows x 4 chunks, chunk c of row r in slot c ^ (r / 2 % 4); 16 headers.
    __device__ __forceinline__ Q4KWide(const Weight &w, int64_t band, int rows, int tile, int lane) {
        base = w.w + (band * (rows / 16) + tile) * 2304;
        sb_stride = w.sb_stride;
        const int r = lane >> 2, n = lane & 15;
        kq = lane >> 4;
        piece_src = 256u + r * 64 + (((lane & 3) ^ ((r >> 1) & 3)) << 4);
        lane4 = lane * 4u;
#pragma unroll
        for (int q = 0; q < 2; q++) piece_at[q] = (kq & 1) * 1024 + n * 64 + (((2 * q + (kq >> 1)) ^ ((n >> 1) & 3)) << 4);
        hdr_at = 2048 + n * 16;
    }
    template <bool ONCE>
    __device__ __forceinline__ void fetch(uint32_t lds, int sb) const {
        const uint8_t *p = base + sb * sb_stride;
        wide_dma16_hint<ONCE>(lds, p, piece_src);
        wide_dma16_hint<ONCE>(lds + 1024, p, piece_src + 1024u);
        wide_dma4(lds + 2048, p, lane4);
    }
    __device__ __forceinline__ void read(Raw &r, const uint8_t *lds, int) const {
        r.hdr = *reinterpret_cast<const uint4 *>(lds + hdr_at);
        r.piece[0] = *reinterpret_cast<const uint4 *>(lds + piece_at[0]);
        r.piece[1] = *reinterpret_cast<const uint4 *>(lds + piece_at[1]);
    }
    // step c = 2 q + nibble plane contracts that plane of chunks 2 q and 2 q + 1: lane kq = 2 * chunk parity + piece takes
    // values 128 q + 64 (kq / 2) + 32 plane + 16 (kq % 2) .. + 15, piece 8 q + 4 (kq / 2) + 2 plane + kq % 2 of a token
    static __device__ __forceinline__ int lane_piece(int kq) { return 4 * (kq >> 1) + (kq & 1); }
    static __device__ constexpr int step_piece(int c) { return 8 * (c >> 1) + 2 * (c & 1); }
    __device__ __forceinline__ void unpack(const Raw &r, Operands &o) const {
        typedef unsigned short us2 __attribute__((ext_vector_type(2)));
        const uint32_t word = (kq & 1) ? (r.hdr.x ^ 0x80000000u) >> 16 : r.hdr.x;
        o.scale = f16_bits_to_f32(word & 0xffffu);
        o.d = f16_bits_to_f32(r.hdr.x & 0xffffu);
        o.dmin = f16_bits_to_f32(r.hdr.x >> 16);
        // runs 4 kq .. + 3 of the activation: the mins of sub-blocks 2 kq and 2 kq + 1, twice each (exact in f16)
        const int odd = 16 * (kq & 1);
        const uint32_t m03 = r.hdr.z >> odd, m47 = ((r.hdr.w >> (odd + 4)) & 0x0f0fu) | ((m03 >> 2) & 0x3030u);
        const uint32_t mw = (kq & 2) ? m47 : m03 & 0x3f3fu;
        const us2 m2 = __builtin_bit_cast(us2, __builtin_amdgcn_perm(mw, mw, 0x0c010c00u));
        const _Float16 ma = static_cast<_Float16>(m2.x), mb = static_cast<_Float16>(m2.y);
        o.mins = v4h_w{ma, ma, mb, mb};
        // scales of chunk 2 q + kq / 2: sub-block 2 * chunk, 2 * chunk + 1
        const int up = 16 * (kq >> 1);
        const uint32_t s03 = r.hdr.y >> up, s47 = ((r.hdr.w >> up) & 0x0f0fu) | ((s03 >> 2) & 0x3030u);
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const uint32_t sc = __builtin_amdgcn_perm(q ? s47 : s03, q ? s47 : s03, 0x0c010c00u);
            const us2 lo = __builtin_bit_cast(us2, sc & 0x00070007u), hi = __builtin_bit_cast(us2, (sc >> 3) & 0x00070007u);
            const uint32_t pc[4] = {r.piece[q].x, r.piece[q].y, r.piece[q].z, r.piece[q].w};
#pragma unroll
            for (int plane = 0; plane < 2; plane++) {  // low nibbles = sub-block 2 * chunk, high = 2 * chunk + 1
                const us2 l2 = plane ? us2{lo.y, lo.y} : us2{lo.x, lo.x}, h2 = plane ? us2{hi.y, hi.y} : us2{hi.x, hi.x};
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const us2 v = __builtin_bit_cast(us2, (pc[m] >> (4 * plane)) & 0x0f0f0f0fu);
                    // (a byte pair times a digit, at most 15 * 7, never carries into its neighbour)
                    o.lo[2 * q + plane][m] = __builtin_bit_cast(int, static_cast<us2>(v * l2));
                    o.hi[2 * q + plane][m] = __builtin_bit_cast(int, static_cast<us2>(v * h2));
                }
            }
        }
    }
    struct Sums {
        v4i_w lo, hi;
        v4f_w p;
    };
    static constexpr int kMfma = 9;
    __device__ __forceinline__ void contract(const Operands &o, const v4i_w (&av)[4], const v4h_w rs, Sums &s) const {
        s.lo = s.hi = v4i_w{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            s.lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[c], o.lo[c], s.lo, 0, 0, 0);
            s.hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[c], o.hi[c], s.hi, 0, 0, 0);
        }
        s.p = __builtin_amdgcn_mfma_f32_16x16x16f16(rs, o.mins, v4f_w{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
    }
    // One matrix instruction forms yd * d and yd * -dmin of two token groups: its four 16 x 16 products of K = 1 are
    // (group 0, d), (group 0, -dmin), (group 1, d), (group 1, -dmin), each the rounded product that a vector multiplication gives.
    static constexpr int kScaleGroups = 2;
    __device__ __forceinline__ void chain(const Sums &s, const v16f_w &y, int g, float (&acc)[4]) const {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[j] = __builtin_fmaf(y[8 * g + 4 + j], s.p[j], acc[j]);
            acc[j] = __builtin_fmaf(y[8 * g + j], static_cast<float>(s.lo[j] + 8 * s.hi[j]), acc[j]);
        }
    }
    __device__ __forceinline__ void chain(const Sums &s, const float (&yv)[4], const Operands &o, float (&acc)[4]) const {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[j] = __builtin_fmaf(-(yv[j] * o.dmin), s.p[j], acc[j]);
            acc[j] = __builtin_fmaf(yv[j] * o.d, static_cast<float>(s.lo[j] + 8 * s.hi[j]), acc[j]);
        }
    }
};

int launch_gemm_q4k_wide(const MatArgs &a, hipStream_t st) {
    return a.group_offsets ? launch_wide_grouped<Q4KWide>(a, st) : launch_wide_plain<Q4KWide>(a, st);
}

}  // namespace cml
