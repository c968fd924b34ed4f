// Asymmetric group-wise 4-bit quantisation of expert weights (load time).
//
// Replaces quantize_w4 (kernels/w4a16.py:19-32), which pack_experts_module /
// _pack_3d (kernels/pack_experts.py:34-41, 87-106) runs per expert on the
// bf16 weights. For each row r and group g of gs consecutive columns, in fp32:
//   wmin, wmax = min, max of the group
//   scale = max(wmax - wmin, 1e-8) / 15
//   zero  = clamp(rint(-wmin / scale), 0, 15)
//   q[k]  = clamp(rint(w[k] / scale + zero), 0, 15)
//   byte j of the row = q[2j] | q[2j+1] << 4;  scale, zero stored as fp16
// rint rounds half to even (torch.round); the divisions are IEEE divisions
// and w / scale + zero is a division then an addition (no fused form), so
// the bytes, scales and zero-points are those of the reference.
//
// The rows' groups follow one another without gaps (K % gs == 0), so the
// kernel sees one list of groups: 16 columns per lane, a group is gs/16
// consecutive lanes of one wave (2, 4 or 8), reduced by DPP lane moves. No
// row is ever looked up.
//
// What bounds it: HBM (2.5 bytes per bf16 weight). The first form (one 4-byte
// load, two divisions and one byte stored per thread, shuffles through LDS)
// was VALU-bound. Here a division is five fused steps on the group's
// reciprocal y (one mul, two residual corrections: Markstein's division, IBM J.
// Res. Dev. 34, 1990), which give the correctly rounded quotient while nothing
// over- or underflows. (The theorem needs y correctly rounded; for a divisor whose
// mantissa is all ones one Newton step does not promise that, but gfx950's estimate
// leads there: tests/test_gpu_load.py, at every such scale's exponent.) d >= 1e-8, and a group with a magnitude of 2^60 or more
// takes the compiler's division; below 2^-102 a residual may be inexact, but
// then the quotient is below 2^-71 and packs as z either way. Not kept: the
// bytes from t = fma(w, y, z) with divisions only near a tie. bf16 weights are
// multiples of a coarse step, so exact ties are common and most waves divided
// (289 against 243 us for gate/up).
// Measured, one layer's bf16 weights (761 M, 1.93 GB in and out): 1454 us (1.3
// TB/s) with the first form, 334 us (5.8 TB/s) with this one.
#include "ksl_common.h"

namespace ksl {
namespace {

constexpr float kDivMax = 0x1p60f;    // largest magnitude of the fused division
constexpr int kQC = 16;               // columns per lane

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));

// Columns 16c .. 16c+15 of the weights as fp32 (exact for every storage type).
// The address is a multiple of a column pair's size only: the vector type says
// so, and global loads need no more than 4 bytes.
template <int DT>
__device__ __forceinline__ void load16(const void* w, int64_t c, float (&v)[kQC]) {
    constexpr int n = DT == KSL_DTYPE_F32 ? 4 : 2;
    const u32x4_a4* p = reinterpret_cast<const u32x4_a4*>(static_cast<const char*>(w) + c * (16 * n));
    u32x4_a4 a[n];
#pragma unroll
    for (int j = 0; j < n; ++j) a[j] = __builtin_nontemporal_load(p + j);
#pragma unroll
    for (int i = 0; i < kQC; ++i) {
        if constexpr (DT == KSL_DTYPE_F32) {
            v[i] = __uint_as_float(a[i >> 2][i & 3]);
        } else {
            const uint32_t u = a[i >> 3][(i >> 1) & 3];
            if constexpr (DT == KSL_DTYPE_F16)
                v[i] = static_cast<float>(__builtin_bit_cast(f16x2, u)[i & 1]);
            else
                v[i] = __uint_as_float(i & 1 ? u & 0xFFFF0000u : u << 16);
        }
    }
}

// The value of a lane's partner: CTRL is a DPP quad permutation or mirror.
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}

// Minimum and maximum over groups of L consecutive lanes (2, 4 or 8).
template <int L>
__device__ __forceinline__ void group_minmax(float& mn, float& mx) {
    mn = fminf(mn, dpp<0xB1>(mn));  // lanes 1, 0, 3, 2
    mx = fmaxf(mx, dpp<0xB1>(mx));
    if constexpr (L >= 4) {
        mn = fminf(mn, dpp<0x4E>(mn));  // lanes 2, 3, 0, 1
        mx = fmaxf(mx, dpp<0x4E>(mx));
    }
    if constexpr (L >= 8) {
        mn = fminf(mn, dpp<0x141>(mn));  // mirror within 8 lanes
        mx = fmaxf(mx, dpp<0x141>(mx));
    }
}

// clamp to [0, 15] by comparisons (torch.clamp's rule: a value equal to a
// bound, -0.0 included, is returned unchanged)
__device__ __forceinline__ float clamp15(float x) { return x < 0.0f ? 0.0f : (x > 15.0f ? 15.0f : x); }

// a / s, correctly rounded (ranges above; a zero may lose its sign), y = 1 / s.
__device__ __forceinline__ float quotient(float a, float s, float y) {
    float q = a * y;
    q = __builtin_fmaf(__builtin_fmaf(-s, q, a), y, q);
    return __builtin_fmaf(__builtin_fmaf(-s, q, a), y, q);
}

// GS: group size. QA: qpacked is 4-byte aligned (else its bytes go out one by one).
template <int DT, int GS, bool QA>
__global__ __launch_bounds__(256) void quantize_w4_kernel(const void* __restrict__ w, int64_t chunks,
                                                          uint8_t* __restrict__ q, f16* __restrict__ scale,
                                                          f16* __restrict__ zero) {
    constexpr int L = GS / kQC;  // lanes of a group
    const int64_t c = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;  // 16-column chunk
    const bool live = c < chunks;  // whole groups: chunks is a multiple of L
    float v[kQC];
    load16<DT>(w, live ? c : 0, v);
    float mn = v[0], mx = v[0];
#pragma unroll
    for (int i = 1; i < kQC; ++i) {
        mn = fminf(mn, v[i]);
        mx = fmaxf(mx, v[i]);
    }
    group_minmax<L>(mn, mx);
    float d = mx - mn;
    d = d < 1e-8f ? 1e-8f : d;
    float s, z;
    uint32_t b[kQC];  // the integer in the low four bits; a NaN weight gives 0
    if (fmaxf(fabsf(mn), fabsf(mx)) < kDivMax) {
        s = quotient(d, 15.0f, 1.0f / 15.0f);
        float y = __builtin_amdgcn_rcpf(s);
        y = __builtin_fmaf(__builtin_fmaf(-s, y, 1.0f), y, y);
        z = clamp15(rintf(copysignf(quotient(-mn, s, y), -mn)));  // -0.0 stays -0.0, as torch.clamp keeps it
#pragma unroll
        for (int i = 0; i < kQC; ++i) {
            const float t = __fadd_rn(quotient(v[i], s, y), z);
            // clamped, the sum with 2^23 rounds half to even and holds the integer
            b[i] = __float_as_uint(__fadd_rn(__builtin_amdgcn_fmed3f(t, 0.0f, 15.0f), 0x1p23f));
        }
    } else {
        s = __fdiv_rn(d, 15.0f);
        z = clamp15(rintf(__fdiv_rn(-mn, s)));
#pragma unroll
        for (int i = 0; i < kQC; ++i) {
            const float t = clamp15(rintf(__fadd_rn(__fdiv_rn(v[i], s), z)));
            b[i] = t > 0.0f ? static_cast<uint32_t>(t) : 0u;
        }
    }
    if (!live) return;
    u32x2_a4 word;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t p[4];  // a column pair in the low byte
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = (b[8 * h + 2 * i + 1] << 4) | b[8 * h + 2 * i];
        const uint32_t lo = __builtin_amdgcn_perm(p[1], p[0], 0x0c0c0400u);  // bytes p0, p1
        const uint32_t hi = __builtin_amdgcn_perm(p[3], p[2], 0x04000c0cu);  // bytes p2, p3 above
        word[h] = lo | hi;
    }
    if constexpr (QA) {
        __builtin_nontemporal_store(word, reinterpret_cast<u32x2_a4*>(q + 8 * c));
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) q[8 * c + i] = static_cast<uint8_t>(word[i >> 2] >> (8 * (i & 3)));
    }
    if ((threadIdx.x & (L - 1)) == 0) {
        scale[c / L] = static_cast<f16>(s);
        zero[c / L] = static_cast<f16>(z);
    }
}

template <int DT, int GS>
void launch_quantize_gs(const void* w, int64_t chunks, uint8_t* q, f16* s, f16* z, hipStream_t st) {
    const dim3 g(static_cast<unsigned>((chunks + 255) / 256)), b(256);
    if (reinterpret_cast<uintptr_t>(q) % 4 == 0)
        hipLaunchKernelGGL((quantize_w4_kernel<DT, GS, true>), g, b, 0, st, w, chunks, q, s, z);
    else
        hipLaunchKernelGGL((quantize_w4_kernel<DT, GS, false>), g, b, 0, st, w, chunks, q, s, z);
}

template <int DT>
int launch_quantize(const void* w, int64_t rows, int64_t K, int64_t gs, uint8_t* q, void* s, void* z,
                    hipStream_t st) {
    const int64_t chunks = rows * (K / kQC);
    if ((rows * (K / 2) + 255) / 256 >= (int64_t(1) << 31)) return KSL_ERR_SHAPE;
    f16* sp = static_cast<f16*>(s);
    f16* zp = static_cast<f16*>(z);
    if (gs == 128) launch_quantize_gs<DT, 128>(w, chunks, q, sp, zp, st);
    else if (gs == 64) launch_quantize_gs<DT, 64>(w, chunks, q, sp, zp, st);
    else if (gs == 32) launch_quantize_gs<DT, 32>(w, chunks, q, sp, zp, st);
    else return KSL_ERR_SHAPE;
    KSL_LAUNCH_CHECK();
    return KSL_OK;
}

// dequant_w4 (kernels/w4a16.py:35-48): W[n, k] = fp16((q - zero) * scale) with
// the difference and the product taken in fp32 (the reference promotes the
// fp16 nibble values against fp32 scale / zero), rounded once to fp16. One
// thread per 8 consecutive K of one row (4 packed bytes in, 16 bytes out);
// group_size % 8 == 0, so the 8 share one (scale, zero).
__global__ __launch_bounds__(256) void dequant_w4_kernel(const uint8_t* __restrict__ q, const f16* __restrict__ scale,
                                                         const f16* __restrict__ zero, int64_t rows, int K, int gs,
                                                         f16* __restrict__ out) {
    const int64_t per_row = K / 8;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= rows * per_row) return;
    const int64_t r = i / per_row;
    const int c8 = static_cast<int>(i - r * per_row) * 8;
    const uint32_t w = *reinterpret_cast<const uint32_t*>(q + r * (K / 2) + c8 / 2);
    const int64_t gi = r * (K / gs) + c8 / gs;
    const float s = static_cast<float>(scale[gi]);
    const float z = static_cast<float>(zero[gi]);
    f16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float qj = static_cast<float>((w >> (4 * j)) & 15u);
        v[j] = static_cast<f16>(__fmul_rn(__fsub_rn(qj, z), s));
    }
    *reinterpret_cast<f16x8*>(out + r * K + c8) = v;
}

}  // namespace
}  // namespace ksl

extern "C" int ksl_dequant_w4(const uint8_t* qpacked, const void* scale, const void* zero, int64_t rows, int64_t K,
                              int64_t group_size, void* out, void* stream) {
    using namespace ksl;
    if (rows < 0 || K <= 0 || group_size <= 0) return KSL_ERR_SHAPE;
    if (group_size % 8 != 0 || K % group_size != 0 || K > (int64_t(1) << 30)) return KSL_ERR_SHAPE;
    if (rows == 0) return KSL_OK;
    if (!qpacked || !scale || !zero || !out) return KSL_ERR_ARG;
    if (reinterpret_cast<uintptr_t>(qpacked) % 4 || reinterpret_cast<uintptr_t>(out) % 16 ||
        reinterpret_cast<uintptr_t>(scale) % 2 || reinterpret_cast<uintptr_t>(zero) % 2)
        return KSL_ERR_ALIGN;
    const int64_t n = rows * (K / 8);
    const int64_t grid = (n + 255) / 256;
    if (grid >= (int64_t(1) << 31)) return KSL_ERR_SHAPE;
    hipLaunchKernelGGL(dequant_w4_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), qpacked, static_cast<const f16*>(scale),
                       static_cast<const f16*>(zero), rows, static_cast<int>(K), static_cast<int>(group_size),
                       static_cast<f16*>(out));
    KSL_LAUNCH_CHECK();
    return KSL_OK;
}

extern "C" int ksl_quantize_w4(const void* w, int w_dtype, int64_t rows, int64_t K, int64_t group_size,
                               uint8_t* qpacked, void* scale, void* zero, void* stream) {
    using namespace ksl;
    if (rows < 0 || K <= 0 || group_size <= 0) return KSL_ERR_SHAPE;
    if (group_size != 32 && group_size != 64 && group_size != 128) return KSL_ERR_SHAPE;
    if (K % group_size != 0 || K > (int64_t(1) << 30)) return KSL_ERR_SHAPE;
    if (rows == 0) return KSL_OK;
    if (!w || !qpacked || !scale || !zero) return KSL_ERR_ARG;
    const int es = w_dtype == KSL_DTYPE_F32 ? 4 : 2;
    if (reinterpret_cast<uintptr_t>(w) % (2 * es) || reinterpret_cast<uintptr_t>(scale) % 2 ||
        reinterpret_cast<uintptr_t>(zero) % 2)
        return KSL_ERR_ALIGN;
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (w_dtype) {
        case KSL_DTYPE_F32: return launch_quantize<KSL_DTYPE_F32>(w, rows, K, group_size, qpacked, scale, zero, st);
        case KSL_DTYPE_F16: return launch_quantize<KSL_DTYPE_F16>(w, rows, K, group_size, qpacked, scale, zero, st);
        case KSL_DTYPE_BF16: return launch_quantize<KSL_DTYPE_BF16>(w, rows, K, group_size, qpacked, scale, zero, st);
    }
    return KSL_ERR_ARG;
}
