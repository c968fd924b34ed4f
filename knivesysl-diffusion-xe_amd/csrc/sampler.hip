// Per-denoising-step sampler pass over [rows, V] logits: entropy, Gumbel-max
// sample and argmax (kernels/fused_sampler_ops.py:22-93), one workgroup per
// row, one read of the row.
//
//   entropy: H = logsumexp(x) - sum(softmax(x) * x), online over the row
//            (running max m, s = sum e^(x-m), t = sum (x-m) e^(x-m)); entries
//            equal to -inf contribute nothing (torch's Categorical.entropy).
//   sample : first index of the max of fp32(x + g), g = -log(-log(u)),
//            u = tl.rand(seed + row, col) clamped to [1e-10, 1 - 1e-7]: Triton's
//            generator, Philox4x32-10 on the counter (col, 0, 0, 0) with the
//            row's key, first output word to float (triton/language/random.py).
//   argmax : first index of the max of x.
// The row goes by in passes of 16 columns per thread (16-byte loads, the next
// pass requested before the current one is worked on). What bounds the step is
// HBM for the entropy and the VALU for the draw: Philox's 16 multiplies and 31
// xors and two logarithms per column were 3/4 of the first form's 173 us at
// [256, 262144]. Columns that cannot win are therefore never drawn:
//  - T, the best noisy score found so far in the row (any wave), is kept in LDS.
//    g <= 15.94, so a column below T - 15.95 cannot reach T and is dropped. Each
//    thread draws its largest column of the first pass before anything else,
//    which brings T near its final value at once.
//  - The others of a wave are collected in LDS (ballot and prefix count) and
//    drawn 128 at a time, two per lane, so no lane idles in the generator.
//  - For a drawn u, g = -log(-log u) <= -log(1 - u): one hardware logarithm of
//    the generator's integer decides whether the exact score can reach T, and
//    only then the two exact logarithms are taken (a few columns per row).
// Whatever is dropped is strictly below a score that the row attains, so the
// result is the first index of the maximum, in any order of the waves. The
// argmax works alike: a pass is searched only where its maximum reaches the
// row's largest value so far. [256, 262144] fp32, undecided rows:
// 173 -> 101 us (entropy alone 48.3 -> 47.5). Of these the stream with entropy
// and argmax takes 48, the collecting about 15 and the generator the rest (42% of
// the columns are drawn on average; 31% would be with T known from the start).
// The per-thread states merge by fixed trees over the lanes and the waves, so
// the entropy does not depend on timing either.
#include "ksl_common.h"

#include <type_traits>

namespace ksl {
namespace {

constexpr int kSmpWaves = 16;
constexpr int kSmpThreads = kSmpWaves * kWave;
constexpr int kCols = 16;              // columns per thread and pass
constexpr int kDraws = 2;                // draws per lane of a collected batch
constexpr int kQueue = kWave * (kDraws + 4);  // collected columns of a wave: less than a batch, and 4 more per lane
constexpr float kGumbelBound = 15.95f;  // > -log(-log(1 - 1e-7)) = 15.94

struct SmpArgs {
    const void* x;
    int64_t stride;  // elements between rows
    int V;
    int64_t seed;
    float* ent;      // [rows] or null
    int64_t* samp;   // [rows] or null (with amax)
    int64_t* amax;   // [rows] or null
};

// One instruction (v_bitop3) for two xors: 120 -> 107 us per step at [256, 262144].
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

// First output words of Philox4x32-10 for N counters (c0[n], 0, 0, 0) and the
// key (k0, k1). The rounds of the N go by together: a round is a chain of a
// multiply and two xors whose latency a few waves do not hide.
template <int N>
__device__ __forceinline__ void philox_first(uint32_t (&c0)[N], uint32_t k0, uint32_t k1) {
    uint32_t c1[N] = {}, c2[N] = {}, c3[N] = {};
#pragma unroll
    for (int r = 0; r < 10; ++r) {
#pragma unroll
        for (int n = 0; n < N; ++n) {
            const uint64_t p0 = static_cast<uint64_t>(0xD2511F53u) * c0[n];
            const uint64_t p2 = static_cast<uint64_t>(0xCD9E8D57u) * c2[n];
            c0[n] = xor3(static_cast<uint32_t>(p2 >> 32), c1[n], k0);
            c2[n] = xor3(static_cast<uint32_t>(p0 >> 32), c3[n], k1);
            c1[n] = static_cast<uint32_t>(p2);
            c3[n] = static_cast<uint32_t>(p0);
        }
        if constexpr (N > 1) __builtin_amdgcn_sched_barrier(0);
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

// Triton's uint32 -> [0, 1): int32 bits, negative i mapped to -i - 1 (= ~i),
// times 4.6566127342e-10 (fp32 0x2fffffff).
__device__ __forceinline__ float uniform_from(uint32_t r) {
    int32_t i = static_cast<int32_t>(r);
    i = i < 0 ? ~i : i;
    return static_cast<float>(i) * __uint_as_float(0x2fffffffu);
}

__device__ __forceinline__ float clamp_uniform(float u) {  // [1e-10, 1 - 1e-7]
    return fminf(fmaxf(u, __uint_as_float(0x2edbe6ffu)), __uint_as_float(0x3f7ffffeu));
}

struct SmpState {
    float m, s, t;     // entropy: running max, sum e^(x-m), sum (x-m) e^(x-m)
    float ab;          // argmax value
    int ai;
    float gb;          // best noisy score
    int gi;
};

// Maximum and minimum over aligned groups of 2^L lanes, by the lane moves of xor_tree_sum.
template <int L, typename T, typename Op>
__device__ __forceinline__ T lane_tree(T v, Op op) {
    static_assert(L == 6 || L == 4);
    const auto bits = [](T x) { return __builtin_bit_cast(uint32_t, x); };
    const auto val = [](uint32_t x) { return __builtin_bit_cast(T, x); };
    if constexpr (L == 6) {
        auto p = __builtin_amdgcn_permlane32_swap(bits(v), bits(v), false, false);
        v = op(val(p[0]), val(p[1]));
        p = __builtin_amdgcn_permlane16_swap(bits(v), bits(v), false, false);
        v = op(val(p[0]), val(p[1]));
    }
    const auto move = [&](auto ctrl, T x) {
        return val(static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(bits(x)), decltype(ctrl)::value, 0xF, 0xF, true)));
    };
    v = op(v, move(std::integral_constant<int, 0x128>{}, v));  // row_ror:8
    v = op(v, move(std::integral_constant<int, 0x140>{}, v));  // mirror within 16 lanes: lane 7 - i of each 8
    v = op(v, move(std::integral_constant<int, 0x4E>{}, v));   // quad_perm [2,3,0,1]
    return op(v, move(std::integral_constant<int, 0xB1>{}, v));
}
template <int L>
__device__ __forceinline__ float lane_max(float v) {
    return lane_tree<L>(v, [](float a, float b) { return fmaxf(a, b); });
}
// The maximum and its lowest index over the group.
template <int L>
__device__ __forceinline__ void lane_argmax(float& b, int& i) {
    const float m = lane_max<L>(b);
    i = lane_tree<L>(b == m ? i : 0x7FFFFFFF, [](int x, int y) { return min(x, y); });
    b = m;
}
// The group's sums relative to its largest maximum.
template <int L>
__device__ __forceinline__ void lane_entropy(float& m, float& s, float& t) {
    const float mn = lane_max<L>(m);
    const float d = m == mn ? 0.0f : fmaxf(m - mn, -200.0f);  // e^-200 is 0; nothing seen: s = t = 0
    const float a = __expf(d);
    t = xor_tree_sum(a * __builtin_fmaf(d, s, t), L);
    s = xor_tree_sum(a * s, L);
    m = mn;
}

// (value, index) maximum, equal values to the lower index.
__device__ __forceinline__ void arg_merge(float& b, int& i, float b2, int i2) {
    if (b2 > b || (b2 == b && i2 < i)) {
        b = b2;
        i = i2;
    }
}

// fp32 as uint32 in the same order (for the LDS maximum), and back.
__device__ __forceinline__ uint32_t ordered(float f) {
    const uint32_t u = __float_as_uint(f);
    return u & 0x80000000u ? ~u : u | 0x80000000u;
}
__device__ __forceinline__ float unordered(uint32_t o) {
    return __uint_as_float(o & 0x80000000u ? o & 0x7FFFFFFFu : ~o);
}

__device__ __forceinline__ float uniform_value(float x) {  // the same in every lane: a scalar register
    return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x)));
}

// Below this a column cannot reach the noisy score T (x + kGumbelBound < T, some ulps to spare).
__device__ __forceinline__ float draw_bound(float T) {
    return T == INFINITY ? T : __builtin_fmaf(fabsf(T), -0x1p-20f, T - kGumbelBound);
}

struct Seen {          // the row's largest values so far, shared by its waves
    uint32_t noisy, plain;
};

// Entropy of 16 columns: x -> the running sums. NaN and -inf contribute nothing.
__device__ __forceinline__ void take_entropy(SmpState& st, const float (&x)[kCols], float gm) {
    constexpr float kLog2e = 1.44269504088896340736f;
    const float mn = fmaxf(st.m, gm);
    const float ref = mn == -INFINITY ? 0.0f : mn;
    const float dm = fmaxf(st.m - ref, -200.0f);  // e^-200 is 0
    const float a = __builtin_amdgcn_exp2f(dm * kLog2e);
    const float s0 = st.s * a, t0 = a * __builtin_fmaf(dm, st.s, st.t);
    float s = s0, t = t0;
#pragma unroll
    for (int i = 0; i < kCols; ++i) {
        const float d = x[i] - ref;
        const float e = __builtin_amdgcn_exp2f(d * kLog2e);
        s += e;
        t = __builtin_fmaf(d, e, t);
    }
    if (!(t == t)) {  // a NaN, or 0 * -inf: of x = -inf, or of a finite x so far below that d overflows
        s = s0;
        t = t0;
#pragma unroll
        for (int i = 0; i < kCols; ++i) {
            // any of these becomes the lowest value, whose e is 0 (so does x = inf: the row ends with s = 0, a NaN)
            const float d = fmaxf(x[i] - ref, -0x1.fffffep127f);
            const float e = __builtin_amdgcn_exp2f(d * kLog2e);
            s += e;
            t = __builtin_fmaf(d, e, t);
        }
    }
    st.m = mn;
    st.s = s;
    st.t = t;
}

// The exact scores of N columns of a lane against its best, of those that can
// reach T. Returns whether any lane of the wave had to look.
template <int N>
__device__ __forceinline__ bool draw(SmpState& st, const float (&x)[N], const int (&col)[N], const bool (&live)[N],
                                     float T, uint32_t k0, uint32_t k1) {
    const float need = __builtin_fmaf(fabsf(T), -0x1p-20f, T - (31 * 0.6931472f + 0.3f));
    uint32_t r[N];
    bool look[N], any = false;
#pragma unroll
    for (int n = 0; n < N; ++n) r[n] = static_cast<uint32_t>(col[n]);
    philox_first<N>(r, k0, k1);
#pragma unroll
    for (int n = 0; n < N; ++n) {
        // u = i 2^-31 for the 31-bit i of r, so g <= -log(1 - u) <= 31 log 2 - log(2^31 - 1 - i)
        // up to the rounding of u (at most 63 of at least 256 steps: 0.29)
        const uint32_t d = (static_cast<uint32_t>(static_cast<int32_t>(r[n]) >> 31) ^ r[n]) ^ 0x7FFFFFFFu;
        const float lim = __builtin_fmaf(__builtin_amdgcn_logf(static_cast<float>(d)), -0.6931472f, x[n]);
        look[n] = live[n] && !(lim < need);
        any = any || look[n];
    }
    if (!__any(any)) return false;
#pragma unroll 1
    for (int n = 0; n < N; ++n)
        if (look[n]) arg_merge(st.gb, st.gi, x[n] + -logf(-logf(clamp_uniform(uniform_from(r[n])))), col[n]);
    return true;
}

template <int XD, bool ENT, bool SAMP>
__global__ __launch_bounds__(kSmpThreads) void sampler_kernel(SmpArgs A) {
    typedef typename Elem<XD>::T XT;
    typedef uint32_t Unit __attribute__((ext_vector_type(4), aligned(4)));  // 16 bytes at any 4-byte address
    constexpr int kN = 16 / static_cast<int>(sizeof(XT));  // columns of a unit
    constexpr int kU = kCols / kN;                         // units per thread and pass
    const int row = blockIdx.x;
    const XT* x0 = static_cast<const XT*>(A.x) + static_cast<int64_t>(row) * A.stride;
    const int tid = threadIdx.x;
    // the row's key: seed + row in int32 when the seed fits int32 (wrapping),
    // else in int64; sign-extended to 64 bits (k0 low, k1 high)
    uint64_t key;
    if (A.seed >= INT32_MIN && A.seed <= INT32_MAX)
        key = static_cast<uint64_t>(static_cast<int64_t>(
            static_cast<int32_t>(static_cast<uint32_t>(A.seed) + static_cast<uint32_t>(row))));
    else
        key = static_cast<uint64_t>(A.seed + row);
    const uint32_t k0 = static_cast<uint32_t>(key), k1 = static_cast<uint32_t>(key >> 32);

    __shared__ SmpState part[kSmpWaves];
    __shared__ Seen seen;
    __shared__ float2 queue[SAMP ? kSmpWaves * kQueue : 1];  // (x, column bits)
    if constexpr (SAMP) {
        if (tid == 0) seen = Seen{ordered(-INFINITY), ordered(-INFINITY)};
        __syncthreads();
    }
    float2* wq = queue + (SAMP ? (tid / kWave) * kQueue : 0);
    int cnt = 0;  // collected columns, the same in every lane

    // columns [0, head) and the last ones one by one, the rest in units of 16
    // bytes from the first 4-byte address
    const int head = (reinterpret_cast<uintptr_t>(x0) & 3) ? 1 : 0;
    const int units = (A.V - head) / kN;
    const int single = A.V - units * kN;
    const Unit* xv = reinterpret_cast<const Unit*>(x0 + head);
    const int passes = (units + kU * kSmpThreads - 1) / (kU * kSmpThreads);
    SmpState st{-INFINITY, 0.0f, 0.0f, -INFINITY, 0, -INFINITY, 0};
    float T = -INFINITY, top = -INFINITY;  // of `seen`, as of the last look
    Unit next[kU];
    if (passes > 0) {
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int i = tid + u * kSmpThreads;
            next[u] = xv[i < units ? i : 0];
        }
    }
    for (int k = 0; k < passes + (single > 0); ++k) {
        float x[kCols];
        int c0, cs;  // column of x[j] : c0 + (j / kN) * cs + j % kN
        if (k < passes) {
            const int i0 = k * (kU * kSmpThreads) + tid;
#pragma unroll
            for (int j = 0; j < kCols; ++j) {
                const uint32_t w = next[j / kN][kN == 4 ? j % kN : (j % kN) / 2];
                if constexpr (XD == KSL_DTYPE_F32) x[j] = __uint_as_float(w);
                else if constexpr (XD == KSL_DTYPE_F16) x[j] = static_cast<float>(__builtin_bit_cast(f16x2, w)[j & 1]);
                else x[j] = __uint_as_float(j & 1 ? w & 0xFFFF0000u : w << 16);
            }
            if ((k + 1) * (kU * kSmpThreads) > units) {  // the last pass: units past the end are NaN, which nothing takes
#pragma unroll
                for (int j = 0; j < kCols; ++j)
                    if (i0 + (j / kN) * kSmpThreads >= units) x[j] = __builtin_nanf("");
            }
            if (k + 1 < passes) {
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    const int i = i0 + (kU + u) * kSmpThreads;
                    next[u] = xv[i < units ? i : 0];
                }
            }
            c0 = head + i0 * kN;
            cs = kSmpThreads * kN;
        } else {
            c0 = tid < head ? tid : units * kN + tid;
            cs = 0;
#pragma unroll
            for (int j = 0; j < kCols; ++j) x[j] = __builtin_nanf("");
            if (tid < single) x[0] = Elem<XD>::load(x0 + c0);
        }
        float gm = -INFINITY;
#pragma unroll
        for (int j = 0; j < kCols; ++j) gm = fmaxf(gm, x[j]);
        if constexpr (ENT) take_entropy(st, x, gm);
        if constexpr (SAMP) {
            const Seen now = seen;
            T = fmaxf(T, uniform_value(unordered(now.noisy)));
            top = fmaxf(top, uniform_value(unordered(now.plain)));
            if (__any(gm >= top)) {
                int best = 0;  // first column of the thread's maximum
#pragma unroll
                for (int j = kCols - 1; j >= 0; --j)
                    if (x[j] == gm) best = c0 + (j / kN) * cs + j % kN;
                arg_merge(st.ab, st.ai, gm, best);
                top = uniform_value(lane_max<6>(st.ab));
                if ((tid & (kWave - 1)) == 0) atomicMax(&seen.plain, ordered(top));
                if (k == 0) {
                    draw<1>(st, {gm}, {best}, {gm > -INFINITY}, T, k0, k1);
                    T = fmaxf(T, uniform_value(lane_max<6>(st.gb)));
                    if ((tid & (kWave - 1)) == 0) atomicMax(&seen.noisy, ordered(T));
                }
            }
            float bound = draw_bound(T);
#pragma unroll
            for (int h = 0; h < kCols; h += 4) {
#pragma unroll
                for (int j = h; j < h + 4; ++j) {
                    const bool in = x[j] >= bound;
                    const uint64_t mask = __ballot(in);
                    if (in) {
                        const int at = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), cnt));
                        wq[at] = make_float2(x[j], __uint_as_float(c0 + (j / kN) * cs + j % kN));
                    }
                    cnt += __popcll(mask);
                }
                const bool last = h + 4 == kCols && k + 1 == passes + (single > 0);
                while (cnt >= kWave * kDraws || (last && cnt > 0)) {
                    const int from = max(cnt - kWave * kDraws, 0);
                    float dx[kDraws];
                    int dc[kDraws];
                    bool live[kDraws];
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int n = 0; n < kDraws; ++n) {
                        const int at = from + n * kWave + (tid & (kWave - 1));
                        live[n] = at < cnt;
                        const float2 e = wq[live[n] ? at : 0];
                        dx[n] = e.x;
                        dc[n] = static_cast<int>(__float_as_uint(e.y));
                    }
                    if (draw<kDraws>(st, dx, dc, live, T, k0, k1)) {
                        T = fmaxf(T, uniform_value(lane_max<6>(st.gb)));
                        bound = draw_bound(T);
                        if ((tid & (kWave - 1)) == 0) atomicMax(&seen.noisy, ordered(T));
                    }
                    cnt = from;
                    __builtin_amdgcn_wave_barrier();
                }
            }
        }
    }
    // merge the lanes of each wave, then the waves: fixed trees
    if constexpr (ENT) lane_entropy<6>(st.m, st.s, st.t);
    if constexpr (SAMP) {
        lane_argmax<6>(st.ab, st.ai);
        lane_argmax<6>(st.gb, st.gi);
    }
    if ((tid & (kWave - 1)) == 0) part[tid / kWave] = st;
    __syncthreads();
    if (tid >= kWave) return;
    SmpState r = part[tid & (kSmpWaves - 1)];
    if constexpr (ENT) lane_entropy<4>(r.m, r.s, r.t);
    if constexpr (SAMP) {
        lane_argmax<4>(r.ab, r.ai);
        lane_argmax<4>(r.gb, r.gi);
    }
    if (tid == 0) {
        if constexpr (ENT) A.ent[row] = logf(r.s) - r.t / r.s;
        if constexpr (SAMP) {
            A.samp[row] = r.gi;
            A.amax[row] = r.ai;
        }
    }
}

template <int XD, bool ENT, bool SAMP>
void launch_smp_x(const SmpArgs& A, int64_t rows, hipStream_t st) {
    hipLaunchKernelGGL((sampler_kernel<XD, ENT, SAMP>), dim3(static_cast<unsigned>(rows)), dim3(kSmpThreads), 0, st, A);
}

template <bool ENT, bool SAMP>
int launch_smp(const void* x, int dtype, int64_t rows, int64_t V, int64_t stride, int64_t seed, float* ent,
               int64_t* samp, int64_t* amax, hipStream_t st) {
    if (rows < 0 || V < 1 || V >= (int64_t(1) << 31) || rows >= (int64_t(1) << 31)) return KSL_ERR_SHAPE;
    if (rows > 0 && stride < V) return KSL_ERR_SHAPE;
    if (rows == 0) return KSL_OK;
    if (!x || (ENT && !ent) || (SAMP && (!samp || !amax))) return KSL_ERR_ARG;
    SmpArgs A{x, stride, static_cast<int>(V), seed, ent, samp, amax};
    switch (dtype) {
        case KSL_DTYPE_F32: launch_smp_x<KSL_DTYPE_F32, ENT, SAMP>(A, rows, st); break;
        case KSL_DTYPE_BF16: launch_smp_x<KSL_DTYPE_BF16, ENT, SAMP>(A, rows, st); break;
        case KSL_DTYPE_F16: launch_smp_x<KSL_DTYPE_F16, ENT, SAMP>(A, rows, st); break;
        default: return KSL_ERR_ARG;
    }
    KSL_LAUNCH_CHECK();
    return KSL_OK;
}

}  // namespace
}  // namespace ksl

extern "C" int ksl_entropy(const void* logits, int dtype, int64_t rows, int64_t V, int64_t row_stride,
                           float* entropy, void* stream) {
    return ksl::launch_smp<true, false>(logits, dtype, rows, V, row_stride, 0, entropy, nullptr, nullptr,
                                        static_cast<hipStream_t>(stream));
}

extern "C" int ksl_gumbel_argmax(const void* logits, int dtype, int64_t rows, int64_t V, int64_t row_stride,
                                 int64_t seed, int64_t* sampled, int64_t* argmax, void* stream) {
    return ksl::launch_smp<false, true>(logits, dtype, rows, V, row_stride, seed, nullptr, sampled, argmax,
                                        static_cast<hipStream_t>(stream));
}

extern "C" int ksl_sample_step(const void* logits, int dtype, int64_t rows, int64_t V, int64_t row_stride,
                               int64_t seed, int64_t* sampled, int64_t* argmax, float* entropy, void* stream) {
    return ksl::launch_smp<true, true>(logits, dtype, rows, V, row_stride, seed, entropy, sampled, argmax,
                                       static_cast<hipStream_t>(stream));
}
