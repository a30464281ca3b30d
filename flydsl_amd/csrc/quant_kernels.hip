// On-device activation quantisers that feed the preshuffle GEMM (gfx950).  HBM-bound elementwise work: each
// input element is read once and each output byte written once.
//
//   psg_launch_quant_pertoken : per-row symmetric quantisation to int8 / OCP e4m3fn + fp32 scale per row
//                               (same results as the host utility: NaN -> 0, +-Inf -> +-dtypeMax, scale = max|row| /
//                               dtypeMax, 1 for an all-zero row, y = x / scale, int8 truncates toward zero, fp8 rounds
//                               to nearest even)
//   psg_launch_quant_mxfp4    : OCP-MX fp4: one e8m0 scale per 32 consecutive K elements (scale byte =
//                               exponent of amax/4 rounded up when its mantissa is >= 1.5), e2m1 codes by nearest
//                               value with ties to the even mantissa, two codes per byte (even k low), scales
//                               written either row-major [R, K/32] or in the shuffled layout the GEMM reads
#include "psg_common.h"

namespace {

enum { X_F32 = 0, X_BF16 = 1, X_F16 = 2 };

template <int XT>
__device__ __forceinline__ void load8(const void* base, size_t elem, float* v) {
    if constexpr (XT == X_F32) {
        const v4f a = *reinterpret_cast<const v4f*>(static_cast<const float*>(base) + elem);
        const v4f b = *reinterpret_cast<const v4f*>(static_cast<const float*>(base) + elem + 4);
        v[0] = a[0]; v[1] = a[1]; v[2] = a[2]; v[3] = a[3]; v[4] = b[0]; v[5] = b[1]; v[6] = b[2]; v[7] = b[3];
    } else {
        const v4i raw = *reinterpret_cast<const v4i*>(static_cast<const uint16_t*>(base) + elem);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t w = (uint32_t)raw[i];
            if constexpr (XT == X_BF16) {
                v[2 * i] = __builtin_bit_cast(float, w << 16);
                v[2 * i + 1] = __builtin_bit_cast(float, w & 0xFFFF0000u);
            } else {
                v[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFF));
                v[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16));
            }
        }
    }
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

// NaN -> 0, +-Inf -> +-dtypeMax, finite values untouched
__device__ __forceinline__ float clean(float t, float dmax) {
    if (t != t) return 0.0f;
    if (__builtin_isinf(t)) return t > 0.0f ? dmax : -dmax;
    return t;
}

// x / s, rounded to nearest even, for a scale s inside [2^-80, 2^100]: y is the correctly rounded 1 / s, so two correction
// steps make the quotient the correctly rounded one (P. Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", 1990: a faithful q, the exact remainder r = x - q s and one more fma).  Inside the bounds a
// remainder can only underflow where |q| < 2^-20, and there every output is a zero; the sign is copied from x because a
// remainder of +0 would turn -0 into +0.  Six instructions for an element against eleven of the IEEE division sequence.
__device__ __forceinline__ float quotient(float x, float s, float y) {
    float q = x * y;
    q = __builtin_fmaf(__builtin_fmaf(-q, s, x), y, q);
    q = __builtin_fmaf(__builtin_fmaf(-q, s, x), y, q);
    return __builtin_copysignf(q, x);
}

template <int OUT_FP8>
__device__ __forceinline__ void quant_store8(const float* q, uint8_t* dst) {
    v2i o;
    if constexpr (OUT_FP8) {
        // v_cvt_pk_fp8_f32: two fp32 -> two OCP e4m3 bytes, round to nearest even (|q| <= 448 here, so its
        // saturation never comes into play)
        unsigned w0 = 0, w1 = 0;
        w0 = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], w0, false);
        w0 = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], w0, true);
        w1 = __builtin_amdgcn_cvt_pk_fp8_f32(q[4], q[5], w1, false);
        w1 = __builtin_amdgcn_cvt_pk_fp8_f32(q[6], q[7], w1, true);
        o[0] = (int)w0;
        o[1] = (int)w1;
    } else {
        uint32_t b[8];
#pragma unroll
        for (int e = 0; e < 8; e++) b[e] = (uint32_t)(int32_t)q[e] & 0xFFu;  // float -> int truncates toward zero
        o[0] = (int)(b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24));
        o[1] = (int)(b[4] | (b[5] << 8) | (b[6] << 16) | (b[7] << 24));
    }
    *reinterpret_cast<v2i*>(dst) = o;
}

// Eight consecutive elements as they are loaded, and what the two passes need of them
typedef unsigned short v2us __attribute__((ext_vector_type(2)));
template <int XT>
struct Raw8 {
    v4i w[XT == X_F32 ? 2 : 1];
    __device__ __forceinline__ void load(const void* base, size_t elem) {
        const v4i* p = reinterpret_cast<const v4i*>(static_cast<const uint8_t*>(base) + elem * (XT == X_F32 ? 4 : 2));
        w[0] = p[0];
        if constexpr (XT == X_F32) w[1] = p[1];
    }
    // running maximum of |x| on the bit patterns, which order like the magnitudes (NaN above Inf above every finite value):
    // fp32 as 32 bits, the 16-bit types as two packed halves
    __device__ __forceinline__ uint32_t max_bits(uint32_t m) const {
#pragma unroll
        for (int j = 0; j < (XT == X_F32 ? 2 : 1); j++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if constexpr (XT == X_F32) {
                    const uint32_t u = (uint32_t)w[j][i] & 0x7FFFFFFFu;
                    m = u > m ? u : m;
                } else {
                    const v2us a = __builtin_bit_cast(v2us, (uint32_t)w[j][i] & 0x7FFF7FFFu), b = __builtin_bit_cast(v2us, m);
                    m = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(a, b));
                }
            }
        return m;
    }
    __device__ __forceinline__ void values(float* v) const {
        if constexpr (XT == X_F32) {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = __int_as_float(w[e >> 2][e & 3]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t u = (uint32_t)w[0][i];
                if constexpr (XT == X_BF16) {
                    v[2 * i] = __builtin_bit_cast(float, u << 16);
                    v[2 * i + 1] = __builtin_bit_cast(float, u & 0xFFFF0000u);
                } else {
                    v[2 * i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u & 0xFFFF));
                    v[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u >> 16));
                }
            }
        }
    }
};

// A row belongs to WPR wavefronts: four (one workgroup of 256 threads per row) or one (four rows per workgroup, nothing to wait
// for at a barrier).  The first KEEP 8-element vectors of every thread stay in registers, as loaded, between the two passes;
// longer rows re-read their tail, which is then still in L2.  Bound: HBM; the first version was bound by its VALU work (about 20
// instructions for an element: NaN / Inf cleaning of every value, IEEE division), so the maximum is taken on packed bit
// patterns, values are only cleaned in rows that hold an Inf or NaN, and the division is quotient().
// Measured, bf16 to fp8, the quantiser and the GEMM behind it: 8192 rows of 4096 132.7 -> 129.9 us (of which the quantiser's
// 100 MB take 20 at the 5.0 TB/s of a large copy), 200 rows of 8192 31.2 -> 29.0; the one-wavefront rows (32768 of 1536) with the
// rest of an MoE layer 932.8 -> 913.6.
template <int XT, int OUT_FP8, int WPR, int KEEP>
__global__ void __launch_bounds__(256) k_quant_pertoken(const void* x, uint8_t* y, float* scale, int M, int K) {
    constexpr int NT = WPR * 64;  // threads of a row
    __shared__ float red[4];
    __shared__ uint32_t redu[4];
    const int wave = wave_id();
    const int row = WPR == 4 ? (int)blockIdx.x : (int)blockIdx.x * 4 + wave;
    if (WPR == 1 && row >= M) return;  // a whole wavefront; no barrier follows
    const int tid = WPR == 4 ? (int)threadIdx.x : (int)(threadIdx.x & 63);
    const float dmax = OUT_FP8 ? 448.0f : 127.0f;
    const size_t base = (size_t)row * (size_t)K;
    const int nvec = K >> 3;  // K % 8 == 0
    Raw8<XT> keep[KEEP];
#pragma unroll
    for (int it = 0; it < KEEP; it++) {
        const int vi = tid + it * NT;
        keep[it].load(x, base + (size_t)(vi < nvec ? vi : 0) * 8);  // threads past the row re-read its first vector: no branch
    }
    uint32_t mb = 0;
#pragma unroll
    for (int it = 0; it < KEEP; it++) mb = keep[it].max_bits(mb);
    for (int vi = tid + KEEP * NT; vi < nvec; vi += NT) {
        Raw8<XT> r;
        r.load(x, base + (size_t)vi * 8);
        mb = r.max_bits(mb);
    }
    if constexpr (XT != X_F32) mb = (mb & 0xFFFFu) > (mb >> 16) ? (mb & 0xFFFFu) : (mb >> 16);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)mb, off, 64);
        mb = o > mb ? o : mb;
    }
    if constexpr (WPR == 4) {
        if ((tid & 63) == 0) redu[wave] = mb;
        __syncthreads();
        const uint32_t a = redu[0] > redu[1] ? redu[0] : redu[1], b = redu[2] > redu[3] ? redu[2] : redu[3];
        mb = a > b ? a : b;
    }
    const bool special = mb >= (XT == X_F32 ? 0x7F800000u : XT == X_BF16 ? 0x7F80u : 0x7C00u);  // the row holds an Inf or NaN
    float amax;
    if (!special) {
        amax = XT == X_F32 ? __builtin_bit_cast(float, mb) : XT == X_BF16 ? __builtin_bit_cast(float, mb << 16) : (float)__builtin_bit_cast(_Float16, (uint16_t)mb);
    } else {
        // NaN counts as 0 and Inf as dtypeMax: the maximum once more, over the cleaned values
        amax = 0.0f;
        for (int vi = tid; vi < nvec; vi += NT) {
            Raw8<XT> r;
            r.load(x, base + (size_t)vi * 8);
            float v[8];
            r.values(v);
#pragma unroll
            for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(clean(v[e], dmax)));
        }
        amax = wave_max(amax);
        if constexpr (WPR == 4) {
            if ((tid & 63) == 0) red[wave] = amax;
            __syncthreads();
            amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        }
    }
    float s = amax / dmax;
    if (s == 0.0f) s = 1.0f;
    if (tid == 0) scale[row] = s;
    const float rs = 1.0f / s;
    const bool exact = !special && s >= 0x1p-80f && s <= 0x1p100f;  // uniform over the row
    auto store = [&](const Raw8<XT>& r, int vi) {
        float v[8];
        r.values(v);
        if (exact) {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = quotient(v[e], s, rs);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = clean(v[e], dmax) / s;
        }
        quant_store8<OUT_FP8>(v, y + base + (size_t)vi * 8);
    };
#pragma unroll
    for (int it = 0; it < KEEP; it++) {
        const int vi = tid + it * NT;
        if (vi < nvec) store(keep[it], vi);
    }
    for (int vi = tid + KEEP * NT; vi < nvec; vi += NT) {
        Raw8<XT> r;
        r.load(x, base + (size_t)vi * 8);
        store(r, vi);
    }
}

// Four consecutive lanes share one 32-element block (8 elements each, so a wavefront reads fully coalesced 16- or
// 32-byte pieces); the block maximum is combined with two lane exchanges.  Rows in [M, R) (padding up to a multiple
// of 32 rows) get scale byte 0 and no codes.
template <int XT>
__global__ void __launch_bounds__(256) k_quant_mxfp4(const void* x, uint8_t* packed, uint8_t* scales, int M, int R, int K,
                                                      int shuffled) {
    const int KB = K >> 5;
    const size_t piece = (size_t)blockIdx.x * 256 + threadIdx.x;  // 8-element piece index over R x K
    const size_t blk = piece >> 2;
    const int sub = (int)(piece & 3);
    const bool live = blk < (size_t)R * KB;
    const int r = live ? (int)(blk / KB) : 0, kb = live ? (int)(blk % KB) : 0;
    float v[8];
    float amax = 0.0f;
    if (live && r < M) {
        load8<XT>(x, (size_t)r * K + (size_t)kb * 32 + sub * 8, v);
#pragma unroll
        for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = 0.0f;
    }
    amax = fmaxf(amax, __shfl_xor(amax, 1, 64));
    amax = fmaxf(amax, __shfl_xor(amax, 2, 64));
    if (!live) return;
    // scale byte: biased exponent of amax/4, +1 when bit 22 is set and (lower mantissa bits or a normal exponent)
    const uint32_t u = __builtin_bit_cast(uint32_t, amax / 4.0f);
    uint32_t e = (u >> 23) & 0xFFu;
    const bool up = (u & 0x400000u) && ((u & 0x3FFFFFu) || e > 0);
    if (e != 0xFFu && up) e = (e + 1) & 0xFFu;
    const float sf = e == 0 ? __builtin_bit_cast(float, 0x00400000u)
                            : (e == 0xFF ? __builtin_bit_cast(float, 0x7F800001u) : __builtin_bit_cast(float, e << 23));
    if (r < M) {
        // v_cvt_scalef32_pk_fp4_f32: (a, b) / scale -> two e2m1 codes (a in the low nibble) into one byte of the word
        unsigned word = 0;
        word = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(word, v[0], v[1], sf, 0);
        word = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(word, v[2], v[3], sf, 1);
        word = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(word, v[4], v[5], sf, 2);
        word = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(word, v[6], v[7], sf, 3);
        *reinterpret_cast<unsigned*>(packed + (size_t)r * (K >> 1) + (size_t)kb * 16 + sub * 4) = word;
    }
    if (sub == 0) {
        size_t off;
        if (shuffled) {
            off = (size_t)(r >> 5) * (32u * (size_t)KB) + (size_t)(kb >> 3) * 256 + (size_t)(kb & 3) * 64 + (size_t)(r & 15) * 4 +
                  (size_t)((kb & 7) >> 2) * 2 + (size_t)((r & 31) >> 4);
        } else {
            off = (size_t)r * KB + kb;
        }
        scales[off] = (uint8_t)e;
    }
}

}  // namespace

hipError_t psg_launch_quant_pertoken(const void* x, int x_dtype, void* y, float* scale, int M, int K, int out_fp8,
                                     hipStream_t stream) {
    // one wavefront per row up to 2048 elements once that still gives every CU two workgroups; else four
    const bool narrow = K <= 2048 && M >= 8 * psg_cu_count();
    const int vec = (K / 8 + (narrow ? 63 : 255)) / (narrow ? 64 : 256);  // vectors per thread
#define PSG_Q4(XT_, F8_, WPR_, KEEP_)                                                                                        \
    hipLaunchKernelGGL((k_quant_pertoken<XT_, F8_, WPR_, KEEP_>), dim3(WPR_ == 4 ? M : (M + 3) / 4), dim3(256), 0, stream, x, \
                       (uint8_t*)y, scale, M, K)
#define PSG_Q3(XT_, F8_)                                                       \
    if (narrow) {                                                              \
        if (vec <= 2) PSG_Q4(XT_, F8_, 1, 2); else PSG_Q4(XT_, F8_, 1, 4);     \
    } else if (vec <= 1) PSG_Q4(XT_, F8_, 4, 1);                               \
    else if (vec <= 2) PSG_Q4(XT_, F8_, 4, 2);                                 \
    else PSG_Q4(XT_, F8_, 4, 4);
#define PSG_Q(XT_) if (out_fp8) { PSG_Q3(XT_, 1) } else { PSG_Q3(XT_, 0) }
    if (x_dtype == X_F32) { PSG_Q(X_F32) } else if (x_dtype == X_BF16) { PSG_Q(X_BF16) } else if (x_dtype == X_F16) { PSG_Q(X_F16) } else return hipErrorInvalidValue;
#undef PSG_Q4
#undef PSG_Q3
#undef PSG_Q
    return hipGetLastError();
}

hipError_t psg_launch_quant_mxfp4(const void* x, int x_dtype, void* packed, void* scales, int M, int R, int K, int shuffled,
                                  hipStream_t stream) {
    const size_t blocks = ((size_t)R * (K / 32) * 4 + 255) / 256;  // four threads per 32-element block
    if (x_dtype == X_F32) hipLaunchKernelGGL((k_quant_mxfp4<X_F32>), dim3(blocks), dim3(256), 0, stream, x, (uint8_t*)packed, (uint8_t*)scales, M, R, K, shuffled);
    else if (x_dtype == X_BF16) hipLaunchKernelGGL((k_quant_mxfp4<X_BF16>), dim3(blocks), dim3(256), 0, stream, x, (uint8_t*)packed, (uint8_t*)scales, M, R, K, shuffled);
    else if (x_dtype == X_F16) hipLaunchKernelGGL((k_quant_mxfp4<X_F16>), dim3(blocks), dim3(256), 0, stream, x, (uint8_t*)packed, (uint8_t*)scales, M, R, K, shuffled);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
