// Q4_K x Q8_K on the wide matrix-core kernel (gemm_wide.hpp): batches of more than 32 tokens, but for small weights whose
// K is cut, and expert groups that hold more than a few assignments each (launch_gemm_q4k_mfma holds the lines).
//
// The integers are those of gemm_q4k_mfma.hip: the 6-bit scale of a sub-block as two 3-bit digits inside the int8 weight
// operand (S = lo + 8 hi, two contractions over the whole super-block), the mins against the sums of the
// activation's 16-value runs in one f16 instruction.  There the 16 operand words of a super-block are formed again for every 64
// tokens and the activation passes through registers on its way to LDS; here once for up to 128.
// Bound: instruction issue, of which a super-block and 16 x 16 cells take nine matrix and 24 vector instructions, and LDS reads (5.5 KB).
// us per launch, before -> after: 14336 x 4096 at 64 / 200 / 512 tokens 19.3 -> 17.8, 54 -> 36, 98 -> 76 (790 TOP/s); 4096 x 14336 at 200 / 512
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
    v4i_w blo[4], bhi[4];
    v4h_w mins;
    float dw, dminw;

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
    __device__ __forceinline__ void fetch(uint32_t lds, int sb) const {
        const uint8_t *p = base + sb * sb_stride;
        wide_dma16(lds, p, piece_src);
        wide_dma16(lds + 1024, p, piece_src + 1024u);
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
    __device__ __forceinline__ void unpack(const Raw &r) {
        typedef unsigned short us2 __attribute__((ext_vector_type(2)));
        uint32_t sc03, sc47, m03, m47;
        q4k_unpack_scales(r.hdr.y, r.hdr.z, r.hdr.w, sc03, sc47, m03, m47);
        dw = f16_bits_to_f32(r.hdr.x & 0xffffu);
        dminw = f16_bits_to_f32(r.hdr.x >> 16);
        // runs 4 kq .. + 3 of the activation: the mins of sub-blocks 2 kq and 2 kq + 1, twice each (exact in f16)
        const uint32_t mw = ((kq & 2) ? m47 : m03) >> (16 * (kq & 1));
        const _Float16 ma = static_cast<_Float16>(static_cast<float>(mw & 0xffu)), mb = static_cast<_Float16>(static_cast<float>((mw >> 8) & 0xffu));
        mins = v4h_w{ma, ma, mb, mb};
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const uint32_t sc = (q ? sc47 : sc03) >> (16 * (kq >> 1));
            const uint32_t dlo = sc & 0x0707u, dhi = (sc >> 3) & 0x0707u;
            const uint32_t pc[4] = {r.piece[q].x, r.piece[q].y, r.piece[q].z, r.piece[q].w};
#pragma unroll
            for (int plane = 0; plane < 2; plane++) {  // low nibbles = sub-block 2 * chunk, high = 2 * chunk + 1
                const us2 l2 = __builtin_bit_cast(us2, __builtin_amdgcn_perm(dlo, dlo, plane ? 0x0c010c01u : 0x0c000c00u));
                const us2 h2 = __builtin_bit_cast(us2, __builtin_amdgcn_perm(dhi, dhi, plane ? 0x0c010c01u : 0x0c000c00u));
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const us2 v = __builtin_bit_cast(us2, (pc[m] >> (4 * plane)) & 0x0f0f0f0fu);
                    // (a byte pair times a digit, at most 15 * 7, never carries into its neighbour)
                    blo[2 * q + plane][m] = __builtin_bit_cast(int, static_cast<us2>(v * l2));
                    bhi[2 * q + plane][m] = __builtin_bit_cast(int, static_cast<us2>(v * h2));
                }
            }
        }
    }
    struct Sums {
        v4i_w lo, hi;
        v4f_w p;
    };
    static constexpr int kMfma = 9, kChainPerMfma = 3;
    __device__ __forceinline__ void contract(const v4i_w (&av)[4], const v4h_w rs, Sums &s) const {
        s.lo = s.hi = v4i_w{0, 0, 0, 0};
        s.p = __builtin_amdgcn_mfma_f32_16x16x16f16(rs, mins, v4f_w{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            s.lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[c], blo[c], s.lo, 0, 0, 0);
            s.hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[c], bhi[c], s.hi, 0, 0, 0);
        }
    }
    __device__ __forceinline__ void chain(const Sums &s, const float (&yv)[4], float (&acc)[4]) const {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            acc[j] = __builtin_fmaf(-(yv[j] * dminw), s.p[j], acc[j]);
            acc[j] = __builtin_fmaf(yv[j] * dw, static_cast<float>(s.lo[j] + 8 * s.hi[j]), acc[j]);
        }
    }
};

int launch_gemm_q4k_wide(const MatArgs &a, hipStream_t st) {
    return a.group_offsets ? launch_wide_grouped<Q4KWide>(a, st) : launch_wide_plain<Q4KWide>(a, st);
}

}  // namespace cml
