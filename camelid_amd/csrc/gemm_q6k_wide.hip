// Q6_K x Q8_K on the wide matrix-core kernel (gemm_wide.hpp): batches of more than 16 tokens, and smaller ones on weights
// of more than 1024 row tiles, but for short rows of tall weights (launch_gemm_q6k_mfma holds the lines).
//
// gemm_q6k_mfma.hip contracts one 16-value sub-block at a time (half of the matrix instruction's K is zero) and
// scales its sums with an integer multiply-add per cell and sub-block: sixteen matrix and 64 vector instructions per
// super-block and 16 x 16 cells.  Here the scale goes into the weight operand: a 6-bit value times its int8
// scale is 13 bits, two int8 bytes, so a super-block is eight full matrix instructions and 16 vector ones per 16 x 16 cells
// (S = lo + 256 hi; then the f32 step), and 180 vector instructions per 16 rows of weight, once for all tokens of the column.
// Bound: instruction issue (a vector instruction 4 cycles, a matrix instruction with 16-byte operands about 8).
// us per launch, before -> after: 4096 x 14336 at 64 / 128 / 512 tokens 41 -> 27, 75 -> 36, 281 -> 80 (751 TOP/s);
// 18944 x 3584 at 16 / 37 / 200 / 512 tokens 21.2 -> 18.5, 44 -> 23, 107 -> 50, 204 -> 91; 128256 x 3072 at 64: 145 -> 104.
#include "gemm_wide.hpp"

#pragma clang fp contract(off)

namespace cml {

int q6k_ksplit_for(int64_t rows, int64_t n_sb);  // gemv_q6k.hip: the matvec kernel's K-split policy

struct Q6KWide {
    static constexpr const char *kName = "q6k";
    static constexpr int kTileBytes = 2048 + 1024 + 256 + 256, kFetches = 5;  // LDS bytes of a wave's super-block (ql | qh | scales | d), requests for it
    static constexpr float kStepUs = 0.30f, kPartUs = 0.18f, kUnpackUs = 0.12f, kCellsUs = 0.12f, kSlabUs = 0.00f;  // (wide_cost)
    static constexpr bool kRunSums = false;
    struct Weight {
        const uint8_t *ql, *qh, *sc, *d;
        int64_t ql_stride, qh_stride, sc_stride, d_stride;
    };
    static Weight weight(const cml_weight *w) {
        return Weight{w->planes.p[0], w->planes.p[1], w->planes.p[2], w->planes.p[3], w->planes.row_stride[0], w->planes.row_stride[1], w->planes.row_stride[2], w->planes.row_stride[3]};
    }
    static int ksplit(int64_t rows, int64_t n_sb) { return q6k_ksplit_for(rows, n_sb); }
    // Lane kq of a row holds bytes 16 kq .. + 15 of the 64 ql bytes of either half h of a super-block: their low nibbles
    // are values 128 h + 16 kq .. + 15 (sub-block 8 h + kq), the high ones values 64 further (sub-block 8 h + 4 + kq).
    // The upper two bits of both sit in bytes 16 (kq % 2) .. of the half's 32 qh bytes, at bits 2 (kq / 2) and 4 + 2 (kq / 2).
    struct Raw {
        uint4 ql[2], qh[2], sc;
        uint32_t d;
    };
    const uint8_t *ql, *qh, *sc, *d;      // of the tile's first row (wave-uniform)
    uint32_t ql_src[2], qh_src, sc_src, d_src;  // where this lane's bytes of the requests lie from there
    int kq, ql_at[2], qh_at[2], n16, d_at, d_odd;
    struct Operands {
        v4i_w lo[4], hi[4];  // the bytes of the values times their sub-block's scale
        float scale;         // d
    };

    // LDS: 16 rows of 128 ql bytes, 16-byte piece p of row r in slot p ^ (r % 8); 16 rows of 64 qh bytes, piece p in slot
    // p ^ (r / 2 % 4); 16 rows of 16 scales; 16 words that hold the rows' d (one of the two halves of an aligned word).
    __device__ __forceinline__ Q6KWide(const Weight &w, int64_t band, int rows, int tile, int lane) {
        const int64_t row0 = band * rows + tile * 16;
        const int last = min(15, rows - 1 - tile * 16);  // rows past the end of the band repeat its last row
        ql = w.ql + row0 * w.ql_stride;
        qh = w.qh + row0 * w.qh_stride;
        sc = w.sc + row0 * w.sc_stride;
        const uint8_t *d0 = w.d + row0 * w.d_stride;  // an even address: its aligned word is fetched
        const int d_off = static_cast<int>(reinterpret_cast<uintptr_t>(d0) & 3);
        d = d0 - d_off;
        const int n = lane & 15;
        kq = lane >> 4;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int r = 8 * i + (lane >> 3);
            ql_src[i] = static_cast<uint32_t>(min(r, last) * static_cast<int>(w.ql_stride)) + (((lane & 7) ^ (r & 7)) << 4);
        }
        const int r4 = lane >> 2;
        qh_src = static_cast<uint32_t>(min(r4, last) * static_cast<int>(w.qh_stride)) + (((lane & 3) ^ ((r4 >> 1) & 3)) << 4);
        sc_src = static_cast<uint32_t>(min(r4, last) * static_cast<int>(w.sc_stride)) + ((lane & 3) << 2);
        d_src = d_off + min(n, last) * static_cast<int>(w.d_stride);
        d_odd = (d_src >> 1) & 1;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            ql_at[h] = n * 128 + (((4 * h + kq) ^ (n & 7)) << 4);
            qh_at[h] = 2048 + n * 64 + (((2 * h + (kq & 1)) ^ ((n >> 1) & 3)) << 4);
        }
        n16 = 3072 + n * 16;
        d_at = 3328 + n * 4;
    }
    template <bool>
    __device__ __forceinline__ void fetch(uint32_t lds, int sb) const {
        wide_dma16(lds, ql + sb * 128, ql_src[0]);
        wide_dma16(lds + 1024, ql + sb * 128, ql_src[1]);
        wide_dma16(lds + 2048, qh + sb * 64, qh_src);
        wide_dma4(lds + 3072, sc + sb * 16, sc_src);
        wide_dma4(lds + 3328, d, (d_src + sb * 2) & ~3u);
    }
    __device__ __forceinline__ void read(Raw &r, const uint8_t *lds, int sb) const {
        r.ql[0] = *reinterpret_cast<const uint4 *>(lds + ql_at[0]);
        r.ql[1] = *reinterpret_cast<const uint4 *>(lds + ql_at[1]);
        r.qh[0] = *reinterpret_cast<const uint4 *>(lds + qh_at[0]);
        r.qh[1] = *reinterpret_cast<const uint4 *>(lds + qh_at[1]);
        r.sc = *reinterpret_cast<const uint4 *>(lds + n16);
        r.d = (*reinterpret_cast<const uint32_t *>(lds + d_at) >> (16 * ((d_odd + sb) & 1))) & 0xffffu;
    }
    // step c = 2 h + nibble plane contracts piece 8 h + 4 plane + kq of the 16 pieces of a token
    static __device__ __forceinline__ int lane_piece(int kq) { return kq; }
    static __device__ constexpr int step_piece(int c) { return 4 * c; }
    // The product of a 6-bit value (code - 32) and its int8 scale needs 13 bits; as p = 256 hi + lo with lo a signed byte
    // both are int8 operands:  r = code * sc + (128 - 32 sc) = p + 128,  hi = r >> 8,  lo = (r & 255) ^ 0x80 as a signed byte.
    // One packed 16-bit multiply-add gives r for two values.
    __device__ __forceinline__ void unpack(const Raw &r, Operands &o) const {
        typedef unsigned short us2 __attribute__((ext_vector_type(2)));
        o.scale = f16_bits_to_f32(r.d);
        const int jj = 2 * (kq >> 1);
        const uint32_t scw[4] = {r.sc.x, r.sc.y, r.sc.z, r.sc.w};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t l[4] = {r.ql[h].x, r.ql[h].y, r.ql[h].z, r.ql[h].w};
            const uint32_t u[4] = {r.qh[h].x, r.qh[h].y, r.qh[h].z, r.qh[h].w};
#pragma unroll
            for (int plane = 0; plane < 2; plane++) {
                const int c = 2 * h + plane;
                const int s = static_cast<int>(scw[c] << (24 - 8 * kq)) >> 24;  // sub-block 8 h + 4 plane + kq
                const uint32_t s2 = __builtin_amdgcn_perm(static_cast<uint32_t>(s), static_cast<uint32_t>(s), 0x01000100u);
                const us2 s16 = __builtin_bit_cast(us2, s2);
                const us2 o16 = s16 * us2{static_cast<unsigned short>(-32), static_cast<unsigned short>(-32)} + us2{128, 128};
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const uint32_t up = (plane ? u[m] >> jj : u[m] << (4 - jj)) & 0x30303030u;
                    uint32_t code = ((plane ? l[m] >> 4 : l[m]) & 0x0f0f0f0fu) | up;
                    asm("" : "+v"(code));  // (the compiler otherwise rebuilds the code for either half of the bytes)
                    const us2 even = __builtin_bit_cast(us2, code & 0x00ff00ffu), odd = __builtin_bit_cast(us2, __builtin_amdgcn_perm(code, code, 0x0c030c01u));
                    const uint32_t re = __builtin_bit_cast(uint32_t, static_cast<us2>(even * s16 + o16));
                    const uint32_t ro = __builtin_bit_cast(uint32_t, static_cast<us2>(odd * s16 + o16));
                    // bytes of values 0..3: even low halves hold values 0 and 2, odd ones 1 and 3
                    o.lo[c][m] = static_cast<int>(__builtin_amdgcn_perm(ro, re, 0x06020400u) ^ 0x80808080u);
                    o.hi[c][m] = static_cast<int>(__builtin_amdgcn_perm(ro, re, 0x07030501u));
                }
            }
        }
    }
    struct Sums {
        v4i_w lo, hi;
    };
    static constexpr int kMfma = 8;
    __device__ __forceinline__ void contract(const Operands &o, const v4i_w (&av)[4], const v4h_w, Sums &s) const {
        s.lo = s.hi = v4i_w{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < 4; c++) {
            s.lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[c], o.lo[c], s.lo, 0, 0, 0);
            s.hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[c], o.hi[c], s.hi, 0, 0, 0);
        }
    }
    static constexpr int kScaleGroups = 0;  // (one multiplication per cell and super-block: not ahead as a matrix instruction)
    __device__ __forceinline__ void chain(const Sums &s, const float (&yv)[4], const Operands &o, float (&acc)[4]) const {
#pragma unroll
        for (int j = 0; j < 4; j++) acc[j] = __builtin_fmaf(o.scale * yv[j], static_cast<float>(s.lo[j] + 256 * s.hi[j]), acc[j]);
    }
};

int launch_gemm_q6k_wide(const MatArgs &a, hipStream_t st) { return launch_wide_plain<Q6KWide>(a, st); }

}  // namespace cml
