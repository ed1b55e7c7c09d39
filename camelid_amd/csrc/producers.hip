// The steps immediately upstream of a quantized projection, fused with the
// activation quantizer so that the f32 intermediate never leaves the chip:
//   rms_norm -> Q8_0 / Q8_K      reference rms_norm_quantize, rms_norm_quantize_q8k
//                                (src/cuda_resident.rs:236-270, :4152-4177), CPU
//                                arithmetic CpuTensor::rms_norm_into, src/tensor/mod.rs:2707-2760
//   silu(gate) * up -> Q8_0/Q8_K reference silu_mul_quantize[_q8k] (src/cuda_resident.rs:
//                                4289-4341), CPU arithmetic CpuTensor::silu_mul,
//                                src/tensor/mod.rs:2610-2634
//   gelu_tanh(gate) * up -> ...  reference geglu_quantize_routed (src/cuda_resident.rs:6301-6343),
//                                CPU arithmetic src/gemma4_runtime.rs:5689-5691
// The quantizers are the ones of quantize.hip (same device functions), so the
// fused result equals the composed one bit for bit.
//
// rms_norm keeps the reference's arithmetic exactly, including the part that
// looks as if it could not be spread over lanes: the squares are summed left to
// right in f32 (a tree sum reassociates and changes greedy tokens, as the
// reference's device lane notes at src/cuda_resident.rs:124-131).
//
// The left-to-right sum in parallel, bit for bit.  While the running sum s stays inside one
// binade 2^E, s is an integer S in [2^23, 2^24) counted in units of ulp = 2^(E-150), and
// s + a rounds to S + round(a / ulp): the increment of a term does not depend on S, except for an
// exact tie (fraction one half), which goes to the even neighbour and so depends on the parity
// of S alone.  A run of terms is therefore a pair (D0, D1): the total increment when the run is
// entered with S even / odd -- and two runs compose like functions, which is associative.
//   1. every thread sums its own contiguous chunk and a workgroup scan gives each chunk an
//      APPROXIMATE incoming sum (any association);
//   2. a chunk whose approximate incoming and outgoing sums, widened by the worst-case
//      difference between any two f32 summation orders, lie in the same binade computes its
//      (D0, D1): it adds its terms, in order, to two values of that binade, one with an even and one
//      with an odd last bit, and takes how far their bits moved (any two sums of one parity move
//      alike); any other chunk (the few where the sum crosses a power of two, the leading ones,
//      anything not finite) is marked for in-order addition;
//   3. neighbouring chunks of the same binade are composed by a segmented scan;
//   4. one wave walks the groups in order: a composed run is applied in O(1) after checking on
//      the EXACT running sum that it enters in the assumed binade and does not leave it (if the
//      check fails the run's terms are added one by one -- the approximation only decides speed,
//      never the result); marked chunks are added term by term as the scalar loop would.
// 4096 values: about 9 marked chunks of 16 terms and as many runs instead of 4096 dependent
// additions.
// Rows are independent: one workgroup per token.  Bound: latency -- a row is one chain of memory, scan and walk, and nearly every
// instruction runs once, so the code itself (4 KB) has to be fetched: short straight phases are worth more than
// parallel ones.  4 or 8 waves where 16 had longer scans and more groups to walk.
#include <atomic>

#include "cml_device.hpp"
#include "cml_host.hpp"

#pragma clang fp contract(off)

namespace cml {

__device__ __forceinline__ float readlane_f32(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// A run of terms as a function of the parity of the sum that enters it.
struct RunPair {
    uint32_t d0, d1;
};
// `left` runs first, then `right`
__device__ __forceinline__ RunPair run_then(const RunPair &left, const RunPair &right) {
    RunPair r;
    r.d0 = left.d0 + ((left.d0 & 1u) ? right.d1 : right.d0);  // (the runs of a group climb through one binade, about 2^23 in all)
    r.d1 = left.d1 + ((left.d1 & 1u) ? right.d0 : right.d1);
    return r;
}

// Segmented inclusive scan over the 64 lanes of a wave: every lane ends up with the composition
// of the runs from its group's first lane to itself, `back` lanes before it.  Rows of 16 lanes by DPP, then row by row
// through lane reads.
__device__ __forceinline__ void run_scan64(RunPair &me, int back, int lane) {
    const int rl = lane & 15, row = lane >> 4;
    auto absorb = [&](uint32_t o0, uint32_t o1, bool take) __attribute__((always_inline)) {
        const RunPair both = run_then(RunPair{o0, o1}, me);
        me.d0 = take ? both.d0 : me.d0;
        me.d1 = take ? both.d1 : me.d1;
    };
    const int in_row = min(rl, back);
    absorb(row_shr_i32<1>(me.d0), row_shr_i32<1>(me.d1), in_row >= 1);
    absorb(row_shr_i32<2>(me.d0), row_shr_i32<2>(me.d1), in_row >= 2);
    absorb(row_shr_i32<4>(me.d0), row_shr_i32<4>(me.d1), in_row >= 4);
    absorb(row_shr_i32<8>(me.d0), row_shr_i32<8>(me.d1), in_row >= 8);
#pragma unroll
    for (int r = 1; r < 4; r++)  // the (by now complete) last lane of row r-1 into row r
        absorb(__builtin_amdgcn_readlane(me.d0, 16 * r - 1), __builtin_amdgcn_readlane(me.d1, 16 * r - 1), row == r && back > rl);
}

// Terms xs[0 .. 4*THREADS*C4) (non-negative f32, zero padded) in LDS, thread t owning the contiguous
// chunk of C4 float4 starting at t*C4.  Returns, in every lane of wave 0, the f32 sum
// (((0 + xs[0]) + xs[1]) + ...) exactly as a scalar loop produces it.  n = number
// of real terms (sets the width of the binade guard).
template <int THREADS, int C4>
__device__ __forceinline__ float ordered_sum_nonneg(const float4 *xs4, int n, int tid) {
    constexpr int kWaves = THREADS / 64;
    __shared__ float s_wave_total[kWaves];
    __shared__ int s_count[kWaves];          // groups per wave
    __shared__ uint4 s_group[kWaves][64];    // in order: binade (0: add in order), D0, D1, first thread | chunks << 16
    const int lane = tid & 63, wave = tid >> 6, row = lane >> 4;
    float4 mine[C4];
#pragma unroll
    for (int j = 0; j < C4; j++) mine[j] = xs4[tid * C4 + j];

    // 1. chunk sums and their exclusive scan (the association of this approximation is free):
    //    rows of 16 lanes by DPP, the three row totals by lane reads
    float local = 0.0f;
#pragma unroll
    for (int j = 0; j < C4; j++) local = local + ((mine[j].x + mine[j].y) + (mine[j].z + mine[j].w));
    float incl = local;
    incl = incl + row_shr_f32<1>(incl);  // lanes at the start of a row receive 0
    incl = incl + row_shr_f32<2>(incl);
    incl = incl + row_shr_f32<4>(incl);
    incl = incl + row_shr_f32<8>(incl);
    const float r0 = readlane_f32(incl, 15), r1 = readlane_f32(incl, 31), r2 = readlane_f32(incl, 47);
    incl = incl + (row == 0 ? 0.0f : (row == 1 ? r0 : (row == 2 ? r0 + r1 : (r0 + r1) + r2)));
    if (lane == 63) s_wave_total[wave] = incl;
    __syncthreads();
    float before = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves - 1; w++) {  // all reads at once, then the additions
        const float tw = s_wave_total[w];
        before = before + (w < wave ? tw : 0.0f);
    }
    const float base = before + (incl - local), after = before + incl;

    // 2. same binade on both sides, with room for the difference between summation orders?
    const float delta = static_cast<float>(n + 64) * 2.384185791015625e-07f;  // (n + 64) * 2^-22
    const uint32_t e_lo = __float_as_uint(base * (1.0f - delta)) >> 23, e_hi = __float_as_uint(after * (1.0f + delta)) >> 23;
    const uint32_t even = __float_as_uint(base) & ~1u, odd = even | 1u;
    float u0 = __uint_as_float(even), u1 = __uint_as_float(odd);
#pragma unroll
    for (int j = 0; j < C4; j++) {
        u0 = u0 + mine[j].x;
        u1 = u1 + mine[j].x;
        u0 = u0 + mine[j].y;
        u1 = u1 + mine[j].y;
        u0 = u0 + mine[j].z;
        u1 = u1 + mine[j].z;
        u0 = u0 + mine[j].w;
        u1 = u1 + mine[j].w;
    }
    const bool run = e_lo == e_hi && e_lo >= 1 && e_lo < 255 && (even >> 23) == e_lo && (__float_as_uint(u0) >> 23) == e_lo && (__float_as_uint(u1) >> 23) == e_lo;
    const int E = run ? static_cast<int>(e_lo) : 0;
    RunPair me{__float_as_uint(u0) - even, __float_as_uint(u1) - odd};

    // 3. compose neighbouring runs of one binade (a wave boundary ends a group; neighbouring in-order chunks form one range)
    const int E_prev = __builtin_amdgcn_update_dpp(0, E, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
    const unsigned long long heads = __ballot(lane == 0 || E_prev != E);
    const int back = lane - (63 - __builtin_clzll(heads & (~0ull >> (63 - lane))));  // to the group's first lane
    run_scan64(me, back, lane);
    // the zero padding behind the last real chunk is not walked at all
    const int n_chunks = (n + 4 * C4 - 1) / (4 * C4);
    const bool tail = tid < n_chunks && (lane == 63 || (heads >> (lane + 1 & 63) & 1) != 0 || tid == n_chunks - 1);
    const unsigned long long tails = __ballot(tail);
    if (lane == 0) s_count[wave] = __builtin_popcountll(tails);
    if (tail) s_group[wave][__builtin_popcountll(tails & ((1ull << lane) - 1ull))] = make_uint4(E, me.d0, me.d1, (tid - back) | (back + 1) << 16);
    __syncthreads();
    if (wave != 0) return 0.0f;

    // 4. the walk, every lane of wave 0 alike.  Lane g first fetches the g-th group of a batch of
    //    up to 64 and, for the case that it is an in-order one, its first chunk, so that the
    //    chain through the running sum reads lanes, not memory.
    float s = 0.0f;
    int cnt_w[kWaves], n_groups = 0;
#pragma unroll
    for (int w = 0; w < kWaves; w++) cnt_w[w] = s_count[w];
#pragma unroll
    for (int w = 0; w < kWaves; w++) n_groups += cnt_w[w];
    n_groups = __builtin_amdgcn_readfirstlane(n_groups);
    for (int g0 = 0; g0 < n_groups; g0 += 64) {
        // the (g0 + lane)-th group: which wave's list, which entry
        int k = g0 + lane, w_mine = 0;
#pragma unroll
        for (int w = 0; w < kWaves - 1; w++) {
            const bool past = w_mine == w && k >= cnt_w[w];
            k -= past ? cnt_w[w] : 0;
            w_mine += past ? 1 : 0;
        }
        const uint4 group = s_group[w_mine][min(k, 63)];  // (lanes past the last group read what nobody looks at)
        const int g_first = min(static_cast<int>(group.w & 0xffffu), THREADS - 1);
        float4 gV[C4];
#pragma unroll
        for (int j = 0; j < C4; j++) gV[j] = xs4[g_first * C4 + j];
        const int here = min(64, n_groups - g0);
        auto add_range = [&](const float4 *p, int chunks) __attribute__((always_inline)) {  // the next chunk read ahead
            float4 next[C4];
#pragma unroll
            for (int j = 0; j < C4; j++) next[j] = p[j];
#pragma unroll 1
            for (int c = 1; c <= chunks; c++) {
                float4 v[C4];
                const float4 *pn = p + min(c, chunks - 1) * C4;
#pragma unroll
                for (int j = 0; j < C4; j++) {
                    v[j] = next[j];
                    next[j] = pn[j];
                }
#pragma unroll
                for (int j = 0; j < C4; j++) {
                    s = s + v[j].x;
                    s = s + v[j].y;
                    s = s + v[j].z;
                    s = s + v[j].w;
                }
            }
        };
        auto add_marked = [&](int g) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < C4; j++) {
                const float x = readlane_f32(gV[j].x, g), y = readlane_f32(gV[j].y, g), z = readlane_f32(gV[j].z, g), w = readlane_f32(gV[j].w, g);
                s = s + x;
                s = s + y;
                s = s + z;
                s = s + w;
            }
            const uint32_t where = __builtin_amdgcn_readlane(group.w, g);
            if ((where >> 16) > 1) add_range(xs4 + ((where & 0xffffu) + 1) * C4, (where >> 16) - 1);
        };
        // A run enters with S even or odd; adding its increment to the BITS of s is adding it
        // to S as long as no carry reaches the exponent field -- which is also the test that
        // the sum stays in the binade.  The tests of a batch are looked at once, behind it.
        const float s_in = s;
        uint32_t off = 0;
        for (int g = 0; g < here; g++) {
            const uint32_t Eg = __builtin_amdgcn_readlane(group.x, g);
            if (Eg == 0) {
                add_marked(g);
            } else {
                const uint32_t D0 = __builtin_amdgcn_readlane(group.y, g), D1 = __builtin_amdgcn_readlane(group.z, g);
                const uint32_t sb = __float_as_uint(s), to = sb + ((sb & 1u) ? D1 : D0);
                off |= (sb ^ (Eg << 23)) | (to ^ (Eg << 23));
                s = __uint_as_float(to);
            }
        }
        if (__builtin_amdgcn_readfirstlane(off) >> 23) {  // the guard was too narrow for this data: still exact
            s = s_in;
            for (int g = 0; g < here; g++) {
                const uint32_t where = __builtin_amdgcn_readlane(group.w, g);
                add_range(xs4 + (where & 0xffffu) * C4, where >> 16);
            }
        }
    }
    return s;
}

// ACT: 0 = f32 output only, 1 = Q8_0, 2 = Q8_K (normed may be written as well), 3 = the row's
// sum of squares alone (into normed[token]).
// Every thread keeps its share of the row in registers (up to kRmsRegs float4) and puts the
// squares into LDS, where ordered_sum_nonneg adds them up; the LDS row is reused for the
// normalised values the quantizers read.
constexpr int kRmsRegs = 4;  // most float4 per thread: rows of up to 4 * 1024 * 4 = 16384 values

template <int ACT, int THREADS, int C4>
__global__ __launch_bounds__(THREADS) void rms_norm_quantize_kernel(const float *__restrict__ x, const float *__restrict__ weight,
                                                                float eps, int cols, float *__restrict__ normed,
                                                                int8_t *__restrict__ q, float *__restrict__ scales) {
    extern __shared__ float4 xs4[];  // the row, padded to whole batches: squares first, then the normalised values
    __shared__ float s_scale;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t token = blockIdx.x;
    const int n4 = cols >> 2;
    const float4 *x4 = reinterpret_cast<const float4 *>(x + token * cols);
    const float4 *w4 = reinterpret_cast<const float4 *>(weight);
    float4 xv[C4], wv[C4];  // (the weight is requested with the row: at the end it would be a second round trip)
#pragma unroll
    for (int k = 0; k < C4; k++) {
        const int i = tid + k * THREADS;
        if (i < n4) xv[k] = x4[i];
    }
    if constexpr (ACT != 3) {
#pragma unroll
        for (int k = 0; k < C4; k++) {
            const int i = tid + k * THREADS;
            if (i < n4) wv[k] = w4[i];
        }
    }
#pragma unroll
    for (int k = 0; k < C4; k++) {
        const int i = tid + k * THREADS;
        if (i < n4) {
            const float4 v = xv[k];
            xs4[i] = make_float4(v.x * v.x, v.y * v.y, v.z * v.z, v.w * v.w);
        }
    }
    // zeros from the end of the row up to THREADS whole chunks: sum + 0 == sum exactly (the sum of
    // squares is never negative) and a zero term has increment 0
    for (int i = n4 + tid; i < THREADS * C4; i += THREADS) xs4[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    __syncthreads();
    const float sum = ordered_sum_nonneg<THREADS, C4>(xs4, cols, tid);  // valid in wave 0
    if constexpr (ACT == 3) {
        if (tid == 0) normed[token] = sum;
        return;
    }
    if (wave == 0) {
        const float mean_square = sum / static_cast<float>(cols);
        if (lane == 0) s_scale = 1.0f / sqrtf(mean_square + eps);
    }
    __syncthreads();
    const float scale = s_scale;
    float4 *n4out = normed ? reinterpret_cast<float4 *>(normed + token * cols) : nullptr;
#pragma unroll
    for (int k = 0; k < C4; k++) {
        const int i = tid + k * THREADS;
        if (i < n4) {
            const float4 v = xv[k], w = wv[k];
            float4 y;
            y.x = (v.x * scale) * w.x;
            y.y = (v.y * scale) * w.y;
            y.z = (v.z * scale) * w.z;
            y.w = (v.w * scale) * w.w;
            if (ACT != 0) xs4[i] = y;
            if (n4out) n4out[i] = y;
        }
    }
    if constexpr (ACT == 0) return;
    __syncthreads();
    uint32_t *q32 = reinterpret_cast<uint32_t *>(q + token * cols);
    if constexpr (ACT == 1) {
        // eight lanes per 32-value block; cols/4 is a multiple of 8, so groups enter and leave together
        float *sc = scales + token * (cols / 32);
        for (int i = tid; i < n4; i += THREADS) {
            float s;
            const uint32_t packed = q8_0_quantize_lane8(xs4[i], s);
            q32[i] = packed;
            if ((i & 7) == 0) sc[i >> 3] = s;
        }
    } else {
        // one wave per 256-value super-block
        float *d = scales + token * (cols / 256);
        for (int sb = wave; sb < cols / 256; sb += THREADS / 64) {
            float dv;
            int bsum;
            const uint32_t packed = q8k_quantize_wave(xs4[sb * 64 + lane], dv, bsum);
            q32[sb * 64 + lane] = packed;
            if (lane == 0) d[sb] = dv;
        }
    }
}

template <int THREADS, int C4>
static int launch_rms_norm(int act, const float *x, const float *weight, float eps, int64_t n_tokens, int cols, float *normed, int8_t *q, float *scales, hipStream_t st) {
    constexpr size_t lds = static_cast<size_t>(THREADS) * C4 * sizeof(float4);  // the row in whole chunks (zero padded)
    constexpr size_t fixed = THREADS / 64 * (64 * sizeof(uint4) + 8) + 16;      // and what the kernel declares: ordered_sum_nonneg's lists, the scale
    static std::atomic<bool> raised{false};
    if (lds + fixed > 64 * 1024 && !raised.load(std::memory_order_acquire)) {  // (a launch may use that much without asking)
        CML_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&rms_norm_quantize_kernel<0, THREADS, C4>), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024));
        CML_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&rms_norm_quantize_kernel<1, THREADS, C4>), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024));
        CML_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&rms_norm_quantize_kernel<2, THREADS, C4>), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024));
        CML_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&rms_norm_quantize_kernel<3, THREADS, C4>), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024));
        raised.store(true, std::memory_order_release);
    }
    const dim3 grid(static_cast<unsigned>(n_tokens)), block(THREADS);
    switch (act) {
        case 0: hipLaunchKernelGGL((rms_norm_quantize_kernel<0, THREADS, C4>), grid, block, lds, st, x, weight, eps, cols, normed, q, scales); break;
        case 1: hipLaunchKernelGGL((rms_norm_quantize_kernel<1, THREADS, C4>), grid, block, lds, st, x, weight, eps, cols, normed, q, scales); break;
        case 3: hipLaunchKernelGGL((rms_norm_quantize_kernel<3, THREADS, C4>), grid, block, lds, st, x, weight, eps, cols, normed, q, scales); break;
        default: hipLaunchKernelGGL((rms_norm_quantize_kernel<2, THREADS, C4>), grid, block, lds, st, x, weight, eps, cols, normed, q, scales); break;
    }
    CML_COUNT_LAUNCH("producer.rms_norm");
    CML_HIP_TRY(hipGetLastError());
    return CML_OK;
}

// `CHUNKS` float4 per thread, the fewest that hold the row; FIRST: the fewest that a row of this workgroup's widths needs.
template <int THREADS, int FIRST, int CHUNKS = kRmsRegs>
static int launch_rms_norm_chunks(int act, const float *x, const float *weight, float eps, int64_t n_tokens, int cols, float *normed, int8_t *q, float *scales, hipStream_t st) {
    if constexpr (CHUNKS > FIRST)
        if (cols <= (CHUNKS - 1) * THREADS * 4) return launch_rms_norm_chunks<THREADS, FIRST, CHUNKS - 1>(act, x, weight, eps, n_tokens, cols, normed, q, scales, st);
    return launch_rms_norm<THREADS, CHUNKS>(act, x, weight, eps, n_tokens, cols, normed, q, scales, st);
}

int launch_rms_norm_quantize(int act, const float *x, const float *weight, float eps, int64_t n_tokens, int64_t cols,
                             float *normed, int8_t *q, float *scales, hipStream_t st) {
    if (n_tokens == 0 || cols == 0) return CML_OK;
    if (cols > static_cast<int64_t>(kRmsRegs) * 1024 * 4)
        return fail(CML_ERR_UNSUPPORTED, "rms_norm row of %lld values exceeds the staging limit of %d", (long long)cols, kRmsRegs * 1024 * 4);
    // us per launch of one row, 256 / 512 / 1024 threads: 2048 values 4.7 / 4.9 / 5.9, 3072 5.4 / 5.4 / 6.6, 4096 6.0 / 5.6 / 7.3, 8192 - / 7.2 / 7.9
    // (512 rows of 4096: 7.9 / 8.0 / 10.5); before, always 1024 threads: 4096 8.0, 512 rows 15.
    const int c = static_cast<int>(cols);
    if (cols <= 3072) return launch_rms_norm_chunks<256, 1, 3>(act, x, weight, eps, n_tokens, c, normed, q, scales, st);
    if (cols <= 4 * kRmsRegs * 512) return launch_rms_norm_chunks<512, 2>(act, x, weight, eps, n_tokens, c, normed, q, scales, st);
    return launch_rms_norm_chunks<1024, 3>(act, x, weight, eps, n_tokens, c, normed, q, scales, st);
}

// h = silu(g) * u = (g / (1 + exp(-g))) * u, quantized on the fly.  Q8_K: one wave per
// 256-value super-block, lane l holding values 4l..4l+3 (the layout of quantize_q8_k_kernel).
// Row r of g / u starts at g + r * in_stride / u + r * in_stride (in_stride = cols for separate
// buffers; 2 * cols with u = g + cols when a fused gate|up projection wrote both halves of a row).
template <int GLU>
__global__ __launch_bounds__(256) void glu_quantize_q8k_kernel(const float *__restrict__ g, const float *__restrict__ u,
                                                               int64_t n_sb, int sb_per_row, int64_t in_stride,
                                                               int8_t *__restrict__ q, float *__restrict__ d) {
    const int lane = threadIdx.x & 63;
    const int64_t sb = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (sb >= n_sb) return;
    const int64_t r = sb / sb_per_row, c = (sb - r * sb_per_row) * 256;
    const float4 v = glu4<GLU>(reinterpret_cast<const float4 *>(g + r * in_stride + c)[lane],
                               reinterpret_cast<const float4 *>(u + r * in_stride + c)[lane]);
    float dv;
    int bsum;
    const uint32_t packed = q8k_quantize_wave(v, dv, bsum);
    reinterpret_cast<uint32_t *>(q + sb * 256)[lane] = packed;
    if (lane == 0) d[sb] = dv;
}

// Q8_0: one thread per 4 values, 8 threads per 32-value block (the layout of quantize_q8_0_kernel).
template <int GLU>
__global__ __launch_bounds__(256) void glu_quantize_q8_0_kernel(const float *__restrict__ g, const float *__restrict__ u,
                                                                int64_t n_blocks, int blocks_per_row, int64_t in_stride,
                                                                int8_t *__restrict__ q, float *__restrict__ scales) {
    const int64_t tid = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const int64_t block = tid >> 3;
    const bool live = block < n_blocks;
    const int64_t bsafe = live ? block : 0;
    const int64_t r = bsafe / blocks_per_row, c = (bsafe - r * blocks_per_row) * 32 + (tid & 7) * 4;
    const float4 v = glu4<GLU>(*reinterpret_cast<const float4 *>(g + r * in_stride + c), *reinterpret_cast<const float4 *>(u + r * in_stride + c));
    float scale;
    const uint32_t packed = q8_0_quantize_lane8(v, scale);
    if (!live) return;
    reinterpret_cast<uint32_t *>(q)[tid] = packed;
    if ((tid & 7) == 0) scales[block] = scale;
}

// glu: 0 = silu, 1 = gelu_tanh; act: 1 = Q8_0, 2 = Q8_K.
int launch_glu_quantize(int glu, int act, const float *g, const float *u, int64_t n_tokens, int64_t cols, int64_t in_stride,
                        int8_t *q, float *scales, hipStream_t st) {
    if (n_tokens == 0 || cols == 0) return CML_OK;
    if (act == 1) {
        const int64_t n_blocks = n_tokens * (cols / 32);
        const dim3 grid(static_cast<unsigned>((n_blocks * 8 + 255) / 256));
        const int bpr = static_cast<int>(cols / 32);
        if (glu == 0) hipLaunchKernelGGL(glu_quantize_q8_0_kernel<0>, grid, dim3(256), 0, st, g, u, n_blocks, bpr, in_stride, q, scales);
        else hipLaunchKernelGGL(glu_quantize_q8_0_kernel<1>, grid, dim3(256), 0, st, g, u, n_blocks, bpr, in_stride, q, scales);
        CML_COUNT_LAUNCH("producer.glu.q8_0");
    } else {
        const int64_t n_sb = n_tokens * (cols / 256);
        const dim3 grid(static_cast<unsigned>((n_sb + 3) / 4));
        const int spr = static_cast<int>(cols / 256);
        if (glu == 0) hipLaunchKernelGGL(glu_quantize_q8k_kernel<0>, grid, dim3(256), 0, st, g, u, n_sb, spr, in_stride, q, scales);
        else hipLaunchKernelGGL(glu_quantize_q8k_kernel<1>, grid, dim3(256), 0, st, g, u, n_sb, spr, in_stride, q, scales);
        CML_COUNT_LAUNCH("producer.glu.q8_k");
    }
    CML_HIP_TRY(hipGetLastError());
    return CML_OK;
}

int launch_silu_mul_quantize(int act, const float *g, const float *u, int64_t n_tokens, int64_t cols, int8_t *q, float *scales,
                             hipStream_t st) {
    return launch_glu_quantize(0, act, g, u, n_tokens, cols, cols, q, scales, st);
}

}  // namespace cml
