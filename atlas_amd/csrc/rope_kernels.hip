// rope_kernels.hip -- per-head QK-RMSNorm fused with half-split RoPE, plain
// half-split RoPE (f32 / f16 storage) and the interleaved operator-API RoPE.
//
// Reference semantics (bisegni/atlas):
//   gemma4_qk_norm_rope_fused_batch_f32   crates/atlas-metal/src/kernels.metal:1098-1142
//   (exact oracle kernel; the _wide variants at :1053-1090, :1151-1195 reorder
//   the sum of squares)
//   Llama half-split RoPE = rope_half_to_interleaved_f32 + rope_f32 +
//   rope_interleaved_to_half_f32   kernels.metal:940-949, 972-994
//   NeuralOps::rope (interleaved) = rope_f32; CPU oracle cpu_rope
//   crates/atlas-ops/tests/phase_02_operators.rs:262-272
//
// QK-norm+RoPE: a "unit" is one (token, head) row of head_dim floats; Q heads
// come first, then the optional single K head.  Wavefronts take units of one
// token (qk_norm_rope_token_kernel, head_dim 64, 128, 256 and 512); any other
// even head_dim, and operands off their vector's alignment, take one wavefront
// per unit with the row in LDS.
#include "device_common.hpp"
#include "launch.hpp"


namespace atlas {
namespace {

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// Token engine (head_dim 64 or 128 P): a wavefront covers units of one token,
// its Q rows and the optional K row after them.  Lane l owns RoPE pairs
// [l*P, l*P + P) of every unit and keeps both halves x[p] and x[p + d/2] in
// registers, so the rotation needs no cross-lane exchange; the token's
// cos/sin row and the four weight slices are loaded once per wavefront.  At
// head_dim 64 a register row holds two units (HPR = 2), one in each half of
// the wavefront.  Loads are straight-line (units past the last are clamped to
// a valid duplicate address, never stored) and nontemporal; squares go to LDS
// and lane u folds unit u in index order (bit-identical to the CPU composition
// rms_norm -> rope).  Every unit is fully read before it is written, so
// q_out == q and k_out == k are allowed.
__device__ __forceinline__ float half_wave_sum_tree_f32(float v) {  // wave_sum_tree_f32's steps inside each 32 lanes
    v = v + dpp_f32<0xb1, 0xf, false>(v);
    v = v + dpp_f32<0x4e, 0xf, false>(v);
    v = v + dpp_f32<0x141, 0xf, false>(v);
    v = v + dpp_f32<0x140, 0xf, false>(v);
    return v + __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401f));
}

template <int P>
struct pvec {
    float v[P];
};

template <int P, bool NT>
__device__ __forceinline__ pvec<P> ld_p(const float* p) {
    constexpr bool nt = NT;
    pvec<P> r;
    if constexpr (P == 1) {
        r.v[0] = nt ? __builtin_nontemporal_load(p) : *p;
    } else if constexpr (P == 2) {
        typedef float f2 __attribute__((ext_vector_type(2)));
        const f2 a = nt ? __builtin_nontemporal_load(reinterpret_cast<const f2*>(p)) : *reinterpret_cast<const f2*>(p);
        r.v[0] = a.x;
        r.v[1] = a.y;
    } else {
        typedef float f4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int j = 0; j < P; j += 4) {
            const f4 a = nt ? __builtin_nontemporal_load(reinterpret_cast<const f4*>(p + j))
                            : *reinterpret_cast<const f4*>(p + j);
            r.v[j] = a.x;
            r.v[j + 1] = a.y;
            r.v[j + 2] = a.z;
            r.v[j + 3] = a.w;
        }
    }
    return r;
}

template <int P>
__device__ __forceinline__ void st_p(float* p, const pvec<P>& r) {
    if constexpr (P == 1) {
        __builtin_nontemporal_store(r.v[0], p);
    } else if constexpr (P == 2) {
        typedef float f2 __attribute__((ext_vector_type(2)));
        __builtin_nontemporal_store(f2{r.v[0], r.v[1]}, reinterpret_cast<f2*>(p));
    } else {
        typedef float f4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int j = 0; j < P; j += 4)
            __builtin_nontemporal_store(f4{r.v[j], r.v[j + 1], r.v[j + 2], r.v[j + 3]},
                                        reinterpret_cast<f4*>(p + j));
    }
}

template <int P>
__device__ __forceinline__ void sq_p(float* dst, const pvec<P>& x) {
#pragma unroll
    for (int j = 0; j < P; ++j) dst[j] = x.v[j] * x.v[j];
}

// MAXU register rows of HPR units per wavefront, WPG wavefronts per
// workgroup; each wavefront uses its own LDS region, so the handoff between
// the lanes that square and the lanes that fold is a wavefront-scope fence,
// not a workgroup barrier.  SPLIT: a token's units are spread over
// consecutive wavefronts, MAXU HPR each; otherwise one wavefront has them all.
// SEQ = false (ATLAS_REDUCTION_WIDE): each unit's sum of squares is a tree sum
// of the lanes' partial sums instead of the in-order fold (no LDS),
// tolerance-level against the CPU operator.
// Parameter order: what the first loads' addresses need (the counts, the
// rows, cos/sin) and epsilon fill the first 56 bytes, which arrive in SGPRs
// at wave launch (kernarg preload); the weights and outputs, needed only
// after the fold, follow.
template <int P, int HPR, int MAXU, int WPG, bool SPLIT, bool SEQ>
__global__ __launch_bounds__(64 * WPG) void qk_norm_rope_token_kernel(
    uint32_t tokens, uint32_t q_heads, uint32_t has_key, uint32_t rope_stride, const float* q, const float* k,
    const float* cosine, const float* sine, float epsilon, const float* q_weight, const float* k_weight,
    float* q_out, float* k_out) {
    constexpr uint32_t kLanes = 64 / HPR;  // lanes of one head row
    constexpr uint32_t HALF = kLanes * P;
    constexpr uint32_t D = 2 * HALF;
    constexpr uint32_t STRIDE = D + 4;
    constexpr uint32_t kUnits = MAXU * HPR;  // a wavefront's units
    // head_dim 256 with one unit per wavefront: the unit's sum by candidate
    // segments (head_fold_candidates), from a padded copy of its squares
    // (float f at f + 4 (f / 64), 68 float4)
    constexpr bool kCand = SEQ && D == 256 && kUnits == 1;
    constexpr uint32_t kLds = kCand ? 272 : (SEQ ? kUnits * STRIDE : 4);
    __shared__ __align__(16) float sq_all[WPG][kLds];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    float* sq = sq_all[wave];
    const uint32_t total = q_heads + has_key;
    const uint32_t wv = blockIdx.x * WPG + wave;
    const uint32_t parts = SPLIT ? (total + kUnits - 1) / kUnits : 1u;
    const uint32_t t = SPLIT ? wv / parts : wv;
    const uint32_t ubase = SPLIT ? (wv - t * parts) * kUnits : 0u;  // the wavefront's first unit
    if (t >= tokens) return;  // wavefront-uniform
    const uint32_t hs = HPR == 1 ? 0u : lane / kLanes;  // the lane's head of each register row
    const uint32_t p0 = (HPR == 1 ? lane : lane % kLanes) * P;

    pvec<P> lo[MAXU], hi[MAXU];
#pragma unroll
    for (int u = 0; u < MAXU; ++u) {
        const uint32_t uu = min(ubase + u * HPR + hs, total - 1);
        const float* src = uu >= q_heads ? k + static_cast<size_t>(t) * D
                                         : q + (static_cast<size_t>(t) * q_heads + uu) * D;
        lo[u] = ld_p<P, true>(src + p0);
        hi[u] = ld_p<P, true>(src + HALF + p0);
    }
    const size_t tb = static_cast<size_t>(t) * rope_stride + p0;
    const pvec<P> c = ld_p<P, false>(cosine + tb);
    const pvec<P> s = ld_p<P, false>(sine + tb);
    const pvec<P> qwl = ld_p<P, false>(q_weight + p0), qwh = ld_p<P, false>(q_weight + HALF + p0);
    const float* kw = has_key ? k_weight : q_weight;
    const pvec<P> kwl = ld_p<P, false>(kw + p0), kwh = ld_p<P, false>(kw + HALF + p0);

    // lane u holds the sum of squares of the wavefront's unit u
    float sum = 0.0f;
    const bool folds = lane < kUnits && ubase + lane < total;
    if constexpr (kCand) {
        // lane l's values p0, p0 + 1 (P = 2) and HALF + p0, ...: each pair
        // inside one 64-float segment
        sq_p<P>(sq + p0 + 4 * (p0 / 64), lo[0]);
        sq_p<P>(sq + HALF + p0 + 4 * ((HALF + p0) / 64), hi[0]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const float f = head_fold_candidates(reinterpret_cast<const f32x4*>(sq), lane);
        sum = lane == 0 ? f : sum;
    } else if constexpr (SEQ) {
#pragma unroll
        for (int u = 0; u < MAXU; ++u) {
            sq_p<P>(sq + (u * HPR + hs) * STRIDE + p0, lo[u]);
            sq_p<P>(sq + (u * HPR + hs) * STRIDE + HALF + p0, hi[u]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // in index order
        if (folds) {
            const f32x4* row = reinterpret_cast<const f32x4*>(sq + lane * STRIDE);
#pragma unroll
            for (uint32_t f = 0; f < D / 4; f += 64)
                sum = fold_lds_chunk(row + f, D / 4 - f < 64 ? D / 4 - f : 64, sum);
        }
    } else {
        (void)sq;
#pragma unroll
        for (int u = 0; u < MAXU; ++u) {
            float part = 0.0f;
#pragma unroll
            for (int j = 0; j < P; ++j) part = part + lo[u].v[j] * lo[u].v[j];
#pragma unroll
            for (int j = 0; j < P; ++j) part = part + hi[u].v[j] * hi[u].v[j];
            if constexpr (HPR == 1) {
                const float f = wave_sum_tree_f32(part);
                sum = lane == static_cast<uint32_t>(u) ? f : sum;
            } else {
                const float f = half_wave_sum_tree_f32(part);
                sum = lane == static_cast<uint32_t>(2 * u) ? readlane_f32(f, 0) : sum;
                sum = lane == static_cast<uint32_t>(2 * u + 1) ? readlane_f32(f, 32) : sum;
            }
        }
    }
    const float inv = folds ? inverse_rms(sum, static_cast<float>(D), epsilon) : 0.0f;

#pragma unroll
    for (int u = 0; u < MAXU; ++u) {
        const uint32_t unit = ubase + u * HPR + hs;
        if (unit < total) {
            // readlane reads the lane's register whatever lanes are active
            float iu = readlane_f32(inv, u * HPR);
            if (HPR == 2) iu = hs ? readlane_f32(inv, u * HPR + 1) : iu;
            const bool key = unit >= q_heads;
            pvec<P> ol, oh;
#pragma unroll
            for (int j = 0; j < P; ++j) {
                const float wl = key ? kwl.v[j] : qwl.v[j];
                const float wh = key ? kwh.v[j] : qwh.v[j];
                const float x0 = lo[u].v[j] * iu * wl;
                const float x1 = hi[u].v[j] * iu * wh;
                ol.v[j] = x0 * c.v[j] - x1 * s.v[j];
                oh.v[j] = x0 * s.v[j] + x1 * c.v[j];
            }
            float* dst = key ? k_out + static_cast<size_t>(t) * D
                             : q_out + (static_cast<size_t>(t) * q_heads + unit) * D;
            st_p<P>(dst + p0, ol);
            st_p<P>(dst + HALF + p0, oh);
        }
    }
}

#define ATLAS_QK_PARAMS                                                                                            \
    hipStream_t stream, const float *q, const float *k, const float *qw, const float *kw, const float *c,          \
        const float *sn, float *qo, float *ko, uint32_t tokens, uint32_t q_heads, uint32_t has_key,                \
        uint32_t rope_stride, float eps
#define ATLAS_QK_ARGS stream, q, k, qw, kw, c, sn, qo, ko, tokens, q_heads, has_key, rope_stride, eps
#define ATLAS_QK_LAUNCH(R, WPG, SPLIT, blocks)                                                                     \
    hipLaunchKernelGGL((qk_norm_rope_token_kernel<P, HPR, R, WPG, SPLIT, SEQ>), dim3(blocks), dim3(64 * (WPG)), 0, \
                       stream, tokens, q_heads, has_key, rope_stride, q, k, c, sn, eps, qw, kw, qo, ko);           \
    return hipGetLastError();

// One wavefront per token (at most 16 units), WPG per workgroup.
template <int P, int HPR, int WPG, bool SEQ>
hipError_t launch_qk_token(ATLAS_QK_PARAMS) {
    const uint32_t rows = (q_heads + has_key + HPR - 1) / HPR, blocks = (tokens + WPG - 1) / WPG;
    if (rows <= 1) { ATLAS_QK_LAUNCH(1, WPG, false, blocks) }
    if (rows <= 2) { ATLAS_QK_LAUNCH(2, WPG, false, blocks) }
    if (rows <= 4) { ATLAS_QK_LAUNCH(4, WPG, false, blocks) }
    if constexpr (HPR == 2) {
        if (rows <= 5) { ATLAS_QK_LAUNCH(5, WPG, false, blocks) }
        ATLAS_QK_LAUNCH(8, WPG, false, blocks)
    } else {
        if (rows <= 8) { ATLAS_QK_LAUNCH(8, WPG, false, blocks) }
        if (rows <= 9) { ATLAS_QK_LAUNCH(9, WPG, false, blocks) }
        if (rows <= 12) { ATLAS_QK_LAUNCH(12, WPG, false, blocks) }
        ATLAS_QK_LAUNCH(16, WPG, false, blocks)
    }
}

// A token's units over several wavefronts, R register rows each, one
// wavefront per workgroup.  (Where one takes them all it is the token form,
// without the division that finds a wavefront's token: 3.42 -> 3.34 us at
// [1000, 1, 256].)
template <int P, int HPR, int R, bool SEQ>
hipError_t launch_qk_split(ATLAS_QK_PARAMS) {
    const uint32_t total = q_heads + has_key;
    if (R < 9 && total <= R * HPR) return launch_qk_token<P, HPR, 1, SEQ>(ATLAS_QK_ARGS);
    ATLAS_QK_LAUNCH(R, 1, true, tokens * ((total + R * HPR - 1) / (R * HPR)))
}

// Units per wavefront by the launch's units (tokens x heads).  A wavefront
// folds its units' rows in order side by side (lane u, unit u), a chain of
// head_dim adds whatever the unit count (64 and three selections for one unit
// at head_dim 256, by candidate segments), while its loads, squares and
// rotations grow with the units it holds: few units are spread over as many
// wavefronts, many are gathered, up to a token's whole row of heads.
// Measured on MI355X (us, graph of back-to-back launches over rotating
// buffers; R = register rows per wavefront, two units each at head_dim 64;
// "token" one wavefront per token; the last column the engine that took 17
// and more heads, and head_dim 64, before):
//   head_dim  units           R=1    R=2    R=4    token or R=9
//   256       2304 (256 x 9)  3.69   3.78   4.34   4.74
//             4352 (256 x 17) 4.44   4.47   4.61   5.35         10.8
//             6912 (768 x 9)  6.10   5.23   5.23   5.73
//             9000 (1000 x 9) 7.18   6.85   5.78   6.07
//             10500 (700 x 15) 8.35  8.10   6.30   7.73
//             13056 (768 x 17) 8.99  8.88   7.56   6.73         14.9
//             34816 (2048 x 17) 19.2 16.8   16.0   13.5         22.9
//   512       1152 (128 x 9)  4.48   5.07   5.32   5.93
//             2048 (128 x 16) 5.44   5.71   6.07   8.15
//             4352 (256 x 17) 7.75   6.29   6.34   7.59         12.8
//             8704 (512 x 17) 11.8   10.4   9.05   8.81         16.8
//   128       1152 (128 x 9)  2.96   3.03   3.30   3.91
//             8704 (512 x 17) 5.13   4.19   4.21   4.70         9.37
//             17000 (1000 x 17) 7.40 6.58   5.24   5.49         12.2
//   64        1280 (256 x 5)  2.50   2.54   2.64   2.79         3.26
//             9000 (1000 x 9) 3.81   3.45   3.65   3.97         5.95
//             36864 (4096 x 9) 7.56  6.79   6.97   5.30         15.9
// From 2048 tokens there are wavefronts enough with one per token, whatever
// its units ([2048, 4 + 1, 256] 6.09 us against 7.44 with four units each),
// four tokens per workgroup ([4096, 8 + 1, 256] 14.17 us against 14.25-14.33
// with one); the tree sum has no chain to spread, so it takes them from 768
// tokens ([1000, 8 + 1, 256] 5.66 against 6.15).  So do tokens of few units
// (to four at head_dim 128, to six wider) from 1200 tokens, which two or four
// to a wavefront divide unevenly (5 as 4 + 1; us, R = 1 / 2 / 4 / token):
//   head_dim 256  3 x 1500  5.13  5.09  4.88  4.74      5 x 1000  -     5.12  -     5.57
//                 5 x 1500  6.75  5.94  6.15  5.75      5 x 2047  7.98  8.22  7.76  6.21
//   head_dim 512  3 x 1250  7.31  6.84  6.32  6.20      3 x 1000  -     6.18  -     6.27
//                 5 x 1500  11.3  10.1  8.93  8.03      5 x 1000  -     -     7.24  7.43
//   head_dim 128  3 x 1750  4.48  4.42  4.04  3.99      6 x 1500  -     -     4.49  4.67
template <int P, int HPR, bool SEQ>
hipError_t launch_qk_p(ATLAS_QK_PARAMS) {
    constexpr uint32_t kOne = P == 4 ? 2100 : (P == 2 ? 4500 : 2500);
    constexpr uint32_t kTwo = P == 4 ? 5000 : (P == 2 ? 7000 : 10000);
    constexpr uint32_t kFour = P == 4 ? 8500 : (P == 2 ? 11000 : 20000);
    constexpr uint32_t kFew = P == 1 ? 4 : 6;
    constexpr uint32_t D = 128 * P / HPR;
    const uint32_t total = q_heads + has_key;
    // a launch's threads are counted in 32 bits: at most 2^26 wavefronts, one
    // per token or, past 16 units, one per 9 register rows
    const uint32_t parts = total > 16 ? (total + 9 * HPR - 1) / (9 * HPR) : 1u;
    const uint32_t most = ((1u << 26) - 8) / parts;
    for (; tokens > most; tokens -= most) {
        const hipError_t e = launch_qk_p<P, HPR, SEQ>(stream, q, k, qw, kw, c, sn, qo, ko, most, q_heads, has_key, rope_stride, eps);
        if (e != hipSuccess) return e;
        if (q_heads) {
            q += static_cast<size_t>(most) * q_heads * D;
            qo += static_cast<size_t>(most) * q_heads * D;
        }
        if (has_key) {
            k += static_cast<size_t>(most) * D;
            ko += static_cast<size_t>(most) * D;
        }
        c += static_cast<size_t>(most) * rope_stride;
        sn += static_cast<size_t>(most) * rope_stride;
    }
    const uint64_t units = static_cast<uint64_t>(tokens) * total;
    if (total <= 16 && tokens >= 2048) return launch_qk_token<P, HPR, 4, SEQ>(ATLAS_QK_ARGS);
    if (total <= 16 && tokens >= 768 && !SEQ) return launch_qk_token<P, HPR, 1, SEQ>(ATLAS_QK_ARGS);
    if (HPR == 1 && total <= kFew && tokens >= 1200) return launch_qk_token<P, HPR, 1, SEQ>(ATLAS_QK_ARGS);
    if (units < kOne) return launch_qk_split<P, HPR, 1, SEQ>(ATLAS_QK_ARGS);
    if (units < kTwo) return launch_qk_split<P, HPR, 2, SEQ>(ATLAS_QK_ARGS);
    if (units < kFour) return launch_qk_split<P, HPR, 4, SEQ>(ATLAS_QK_ARGS);
    if (total > 16) return launch_qk_split<P, HPR, 9, SEQ>(ATLAS_QK_ARGS);
    return launch_qk_token<P, HPR, 1, SEQ>(ATLAS_QK_ARGS);
}
#undef ATLAS_QK_LAUNCH

// Generic fallback (other even head_dims, unaligned operands): one wave per
// unit, row staged in LDS.
__global__ __launch_bounds__(64) void qk_norm_rope_generic_kernel(
    const float* q, const float* k, const float* q_weight, const float* k_weight,
    const float* cosine, const float* sine, float* q_out, float* k_out, uint32_t tokens,
    uint32_t q_heads, uint32_t has_key, uint32_t head_dim, uint32_t rope_stride, float epsilon,
    int sequential) {
    extern __shared__ float row[];
    __shared__ float inv_shared;
    const uint32_t lane = threadIdx.x;
    const uint32_t total = q_heads + has_key;
    const uint32_t unit = blockIdx.x;
    if (unit >= tokens * total) return;
    const uint32_t t = unit / total, local = unit % total;
    const bool key = local >= q_heads;
    const float* src = key ? k + static_cast<size_t>(t) * head_dim
                           : q + (static_cast<size_t>(t) * q_heads + local) * head_dim;
    float* dst = key ? k_out + static_cast<size_t>(t) * head_dim
                     : q_out + (static_cast<size_t>(t) * q_heads + local) * head_dim;
    const float* w = key ? k_weight : q_weight;
    float partial = 0.0f;
    for (uint32_t i = lane; i < head_dim; i += kWave) {
        float v = src[i];
        row[i] = v;
        partial = partial + v * v;
    }
    __syncthreads();
    float inv;
    if (sequential) {
        if (lane == 0) {
            float s = 0.0f;
            for (uint32_t i = 0; i < head_dim; ++i) s = s + row[i] * row[i];
            inv_shared = inverse_rms(s, static_cast<float>(head_dim), epsilon);
        }
        __syncthreads();
        inv = inv_shared;
    } else {
        inv = inverse_rms(wave_sum(partial), static_cast<float>(head_dim), epsilon);
    }
    const uint32_t half = head_dim / 2;
    for (uint32_t p = lane; p < half; p += kWave) {
        const float x0 = row[p] * inv * w[p];
        const float x1 = row[p + half] * inv * w[p + half];
        const float c = cosine[static_cast<size_t>(t) * rope_stride + p];
        const float s = sine[static_cast<size_t>(t) * rope_stride + p];
        dst[p] = x0 * c - x1 * s;
        dst[p + half] = x0 * s + x1 * c;
    }
}

// Half-split RoPE.  Each thread rotates P consecutive pairs of one
// (token, head): x[p..p+P) and x[p+d/2..p+d/2+P) with cos/sin[t*stride + p..]
// -- 128-bit accesses for the vector forms (P = 4 f32, P = 8 f16),
// nontemporal for the streamed rows, cached for the per-token tables that
// every head of the token reuses.
template <int P>
__device__ __forceinline__ void ld_tab(const float* p, float* dst) {
    if constexpr (P % 4 == 0) {
#pragma unroll
        for (int j = 0; j < P; j += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(p + j);
            dst[j] = v.x;
            dst[j + 1] = v.y;
            dst[j + 2] = v.z;
            dst[j + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < P; ++j) dst[j] = p[j];
    }
}

// One thread's P pairs (starting at pair p) of one (token t, head) unit of a
// [tokens, heads, head_dim] tensor; `unit` = t * heads + head.
template <int P>
__device__ __forceinline__ void rope_half_f32_unit(const float* x, const float* cosine, const float* sine,
                                                   float* out, uint64_t unit, uint32_t p, uint32_t t,
                                                   uint32_t head_dim, uint32_t rope_stride) {
    const uint32_t half = head_dim / 2;
    const size_t base = unit * head_dim;
    float a[P], b[P], c[P], s[P];
    if constexpr (P == 4) {
        const f32x4 va = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(x + base + p));
        const f32x4 vb = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(x + base + p + half));
        a[0] = va.x; a[1] = va.y; a[2] = va.z; a[3] = va.w;
        b[0] = vb.x; b[1] = vb.y; b[2] = vb.z; b[3] = vb.w;
    } else {
        a[0] = x[base + p];
        b[0] = x[base + p + half];
    }
    const size_t tb = static_cast<size_t>(t) * rope_stride + p;
    ld_tab<P>(cosine + tb, c);
    ld_tab<P>(sine + tb, s);
    float o0[P], o1[P];
#pragma unroll
    for (int j = 0; j < P; ++j) {
        o0[j] = a[j] * c[j] - b[j] * s[j];
        o1[j] = a[j] * s[j] + b[j] * c[j];
    }
    if constexpr (P == 4) {
        __builtin_nontemporal_store(f32x4{o0[0], o0[1], o0[2], o0[3]}, reinterpret_cast<f32x4*>(out + base + p));
        __builtin_nontemporal_store(f32x4{o1[0], o1[1], o1[2], o1[3]},
                                    reinterpret_cast<f32x4*>(out + base + p + half));
    } else {
        out[base + p] = o0[0];
        out[base + p + half] = o1[0];
    }
}

typedef uint32_t u32x4r __attribute__((ext_vector_type(4)));

template <int P>
__device__ __forceinline__ void rope_half_f16_unit(const uint16_t* x, const float* cosine, const float* sine,
                                                   uint16_t* out, uint64_t unit, uint32_t p, uint32_t t,
                                                   uint32_t head_dim, uint32_t rope_stride) {
    const uint32_t half = head_dim / 2;
    const size_t base = unit * head_dim;
    uint16_t a[P], b[P];
    if constexpr (P == 8) {
        const u32x4r va = __builtin_nontemporal_load(reinterpret_cast<const u32x4r*>(x + base + p));
        const u32x4r vb = __builtin_nontemporal_load(reinterpret_cast<const u32x4r*>(x + base + p + half));
        const uint32_t wa[4] = {va.x, va.y, va.z, va.w}, wb[4] = {vb.x, vb.y, vb.z, vb.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            a[2 * j] = static_cast<uint16_t>(wa[j]);
            a[2 * j + 1] = static_cast<uint16_t>(wa[j] >> 16);
            b[2 * j] = static_cast<uint16_t>(wb[j]);
            b[2 * j + 1] = static_cast<uint16_t>(wb[j] >> 16);
        }
    } else {
        a[0] = x[base + p];
        b[0] = x[base + p + half];
    }
    const size_t tb = static_cast<size_t>(t) * rope_stride + p;
    float c[P], s[P];
    ld_tab<P>(cosine + tb, c);
    ld_tab<P>(sine + tb, s);
    uint16_t o0[P], o1[P];
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const float x0 = h2f(a[j]), x1 = h2f(b[j]);
        o0[j] = f2h(x0 * c[j] - x1 * s[j]);
        o1[j] = f2h(x0 * s[j] + x1 * c[j]);
    }
    if constexpr (P == 8) {
        u32x4r r0, r1;
        r0.x = o0[0] | (static_cast<uint32_t>(o0[1]) << 16);
        r0.y = o0[2] | (static_cast<uint32_t>(o0[3]) << 16);
        r0.z = o0[4] | (static_cast<uint32_t>(o0[5]) << 16);
        r0.w = o0[6] | (static_cast<uint32_t>(o0[7]) << 16);
        r1.x = o1[0] | (static_cast<uint32_t>(o1[1]) << 16);
        r1.y = o1[2] | (static_cast<uint32_t>(o1[3]) << 16);
        r1.z = o1[4] | (static_cast<uint32_t>(o1[5]) << 16);
        r1.w = o1[6] | (static_cast<uint32_t>(o1[7]) << 16);
        __builtin_nontemporal_store(r0, reinterpret_cast<u32x4r*>(out + base + p));
        __builtin_nontemporal_store(r1, reinterpret_cast<u32x4r*>(out + base + p + half));
    } else {
        out[base + p] = o0[0];
        out[base + p + half] = o1[0];
    }
}

// Interleaved pairs (NeuralOps::rope): out[2p] = x0*c - x1*s, out[2p+1] = x0*s + x1*c,
// one cos/sin row shared by every input row.
__global__ __launch_bounds__(256) void rope_interleaved_kernel(const float* x, const float* cosine,
                                                               const float* sine, float* out,
                                                               uint32_t rows, uint32_t hidden) {
    const uint32_t pairs = hidden / 2;
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<uint64_t>(rows) * pairs) return;
    const uint32_t p = static_cast<uint32_t>(i % pairs);
    const size_t b = (i / pairs) * hidden + 2 * p;
    const float x0 = x[b], x1 = x[b + 1];
    const float c = cosine[p], s = sine[p];
    const float o0 = x0 * c - x1 * s;
    const float o1 = x0 * s + x1 * c;
    out[b] = o0;
    out[b + 1] = o1;
}

bool aligned(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

}  // namespace

hipError_t launch_qk_norm_rope_f32(hipStream_t stream, Reduction red, const float* q, const float* k,
                                   const float* q_weight, const float* k_weight,
                                   const float* cosine, const float* sine, float* q_out,
                                   float* k_out, uint32_t tokens, uint32_t q_heads,
                                   uint32_t has_key, uint32_t head_dim, uint32_t rope_stride,
                                   float epsilon) {
    // the rotation after the norm can cancel, so only ATLAS_REDUCTION_WIDE
    // reorders the sum of squares here; kAuto keeps the sequential fold
    const bool seq = red != kWide;
    // Token engine: head_dim 64 or 128*P, operands and per-token cos/sin rows
    // aligned to P floats; the in-order fold, or under WIDE the wavefront
    // tree sum.
    const uint32_t P = head_dim == 64 ? 1 : head_dim / 128;
    const uintptr_t pa = 4u * (P == 0 ? 1 : P);
    const bool ok = (head_dim == 64 || (head_dim % 128 == 0 && (P == 1 || P == 2 || P == 4))) && aligned(q, pa) &&
                    aligned(q_out, pa) && aligned(q_weight, pa) && aligned(cosine, pa) && aligned(sine, pa) &&
                    rope_stride % P == 0 &&
                    (!has_key || (aligned(k, pa) && aligned(k_out, pa) && aligned(k_weight, pa)));
    if (ok) {
        const float *qw = q_weight, *kw = k_weight, *c = cosine, *sn = sine;
        float *qo = q_out, *ko = k_out;
        const float eps = epsilon;
#define ATLAS_QK_P(PP, HPR) \
    return seq ? launch_qk_p<PP, HPR, true>(ATLAS_QK_ARGS) : launch_qk_p<PP, HPR, false>(ATLAS_QK_ARGS);
        if (head_dim == 64) { ATLAS_QK_P(1, 2) }
        if (P == 1) { ATLAS_QK_P(1, 1) }
        if (P == 2) { ATLAS_QK_P(2, 1) }
        ATLAS_QK_P(4, 1)
#undef ATLAS_QK_P
    }
    const uint32_t units = tokens * (q_heads + has_key);
    hipLaunchKernelGGL(qk_norm_rope_generic_kernel, dim3(units), dim3(kWave),
                       static_cast<size_t>(head_dim) * sizeof(float), stream, q, k, q_weight,
                       k_weight, cosine, sine, q_out, k_out, tokens, q_heads, has_key, head_dim,
                       rope_stride, epsilon, seq ? 1 : 0);
    return hipGetLastError();
}

// Two tensors sharing the cos/sin rows (Q and K of the same tokens): threads
// [0, tokens*heads0*groups) rotate x0, the following ones x1; heads1 = 0
// rotates one tensor.  Parameters in kernarg-preload order: the counts, the inputs and
// cos/sin fill the first 56 bytes (user SGPRs at wave launch), the outputs
// follow.
template <int P>
__global__ __launch_bounds__(256) void rope_half_f32_kernel(uint32_t tokens, uint32_t head_dim,
                                                            uint32_t rope_stride, uint32_t heads0, uint32_t heads1,
                                                            const float* x0, const float* x1, const float* cosine,
                                                            const float* sine, float* out0, float* out1) {
    const uint32_t groups = (head_dim / 2) / P;
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x;  // 256-thread workgroups
    const uint64_t total0 = static_cast<uint64_t>(tokens) * heads0 * groups;
    const uint64_t total1 = static_cast<uint64_t>(tokens) * heads1 * groups;
    const bool second = i >= total0;
    if (second && i - total0 >= total1) return;
    const uint64_t j = second ? i - total0 : i;
    const uint64_t unit = j / groups;
    const uint32_t t = static_cast<uint32_t>(unit / (second ? heads1 : heads0));
    const uint32_t p = static_cast<uint32_t>(j - unit * groups) * P;
    if (second)
        rope_half_f32_unit<P>(x1, cosine, sine, out1, unit, p, t, head_dim, rope_stride);
    else
        rope_half_f32_unit<P>(x0, cosine, sine, out0, unit, p, t, head_dim, rope_stride);
}

template <int P>
__global__ __launch_bounds__(256) void rope_half_f16_kernel(uint32_t tokens, uint32_t head_dim,
                                                            uint32_t rope_stride, uint32_t heads0, uint32_t heads1,
                                                            const uint16_t* x0, const uint16_t* x1, const float* cosine,
                                                            const float* sine, uint16_t* out0, uint16_t* out1) {
    const uint32_t groups = (head_dim / 2) / P;
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x;  // 256-thread workgroups
    const uint64_t total0 = static_cast<uint64_t>(tokens) * heads0 * groups;
    const uint64_t total1 = static_cast<uint64_t>(tokens) * heads1 * groups;
    const bool second = i >= total0;
    if (second && i - total0 >= total1) return;
    const uint64_t j = second ? i - total0 : i;
    const uint64_t unit = j / groups;
    const uint32_t t = static_cast<uint32_t>(unit / (second ? heads1 : heads0));
    const uint32_t p = static_cast<uint32_t>(j - unit * groups) * P;
    if (second)
        rope_half_f16_unit<P>(x1, cosine, sine, out1, unit, p, t, head_dim, rope_stride);
    else
        rope_half_f16_unit<P>(x0, cosine, sine, out0, unit, p, t, head_dim, rope_stride);
}

// Token engine for the half-split rotation: one wavefront per token covers
// every head of both tensors.  A head row of d elements is 2G 16-byte
// vectors (G = (d/2)/V, V = 8 halves or 4 floats); lane l holds vector
// c = l mod 2G of heads l/2G, l/2G + 64/2G, ..., so each load and store
// instruction covers whole consecutive rows.  Lanes c < G hold x[p] (first
// half), lanes c >= G hold x[p + d/2]; the partner vector sits in lane l ^ G
// and is exchanged with one cross-lane shuffle per dword.  The token's
// cos/sin group (pairs [(c mod G)V, +V)) is loaded once per lane and reused by
// all its heads.  Every head's loads are issued before the first rotation
// (NI head steps per lane, clamped to a valid head and never stored past the
// end).  Same roundings as rope_half_f*_unit: (x0*c) - (x1*s) for the first
// half, (x0*s) + (x1*c) for the second.
//
// GSH = log2(G) when it is 2 or 3 (G = 4: f16 head_dim 64; G = 8: f32
// head_dim 64, f16 head_dim 128): the lanes of the second half hold their
// vectors in reverse order (lane G + j holds vector 2G - 1 - j), so a lane's
// partner is its mirror within the 2G-lane group and the exchange is one
// DPP move per dword (row_half_mirror / row_mirror) instead of a cross-lane
// shuffle through the LDS crossbar.  GSH = -1: G from g_shift at run time,
// natural order, shuffle exchange.
template <int GSH>
__device__ __forceinline__ uint32_t rope_partner(uint32_t own, uint32_t G) {
    if constexpr (GSH == 2)
        return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(own), 0x141, 0xf, 0xf, false));
    else if constexpr (GSH == 3)
        return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(own), 0x140, 0xf, 0xf, false));
    else
        return static_cast<uint32_t>(__shfl_xor(static_cast<int>(own), static_cast<int>(G), kWave));
}

// Parameter order: the counts, the input rows and cos/sin fill the first 56
// bytes, which arrive in SGPRs at wave launch (kernarg preload); the
// outputs, needed only at the stores, follow.
template <bool F16, int NI, int GSH>
__global__ __launch_bounds__(256) void rope_half_token_kernel(uint32_t tokens, uint32_t head_dim, uint32_t heads0,
                                                              uint32_t heads1, uint32_t rope_stride,
                                                              uint32_t g_shift_rt, const uint8_t* x0,
                                                              const uint8_t* x1, const float* cosine,
                                                              const float* sine, uint8_t* out0, uint8_t* out1) {
    constexpr uint32_t V = F16 ? 8 : 4;
    constexpr uint32_t kEsz = F16 ? 2 : 4;
    constexpr bool kMirror = GSH >= 0;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= tokens) return;
    const uint32_t g_shift = kMirror ? static_cast<uint32_t>(GSH) : g_shift_rt;
    const uint32_t G = 1u << g_shift;
    const uint32_t c = lane & (2 * G - 1), hl = lane >> (g_shift + 1);
    const bool first = c < G;
    // the vector of the head row this lane holds, and its pair group
    const uint32_t vec = first || !kMirror ? c : 3 * G - 1 - c;
    const uint32_t g = vec & (G - 1);
    const uint32_t hps = 32u >> g_shift;  // heads per step
    const uint32_t heads = heads0 + heads1;
    const size_t row_bytes = static_cast<size_t>(head_dim) * kEsz;
    float cs[V], sn[V];
    ld_tab<V>(cosine + static_cast<size_t>(t) * rope_stride + g * V, cs);
    ld_tab<V>(sine + static_cast<size_t>(t) * rope_stride + g * V, sn);
    // Both halves as one form, y = own*c + par*s' with s' = -s on the first
    // half's lanes: x0*c - x1*s is x0*c + x1*(-s) (IEEE subtraction adds the
    // negation, and round-to-nearest is symmetric in sign, so fl(x1*(-s)) =
    // -fl(x1*s), zeros included), and x0*s + x1*c is x1*c + x0*s (addition
    // commutes).  No per-value select between the halves' formulas.
#pragma unroll
    for (int j = 0; j < static_cast<int>(V); ++j) sn[j] = first ? -sn[j] : sn[j];
    // row offset of head step i (clamped to a valid head for the load; a step
    // past the last head is never stored, so the store reuses the offset)
    size_t off[NI];
    bool sec[NI];
    u32x4r v[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const uint32_t h = min(hl + static_cast<uint32_t>(i) * hps, heads - 1);
        sec[i] = h >= heads0;
        off[i] = (sec[i] ? static_cast<size_t>(t) * heads1 + (h - heads0) : static_cast<size_t>(t) * heads0 + h) *
                     row_bytes + vec * 16u;
        v[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4r*>((sec[i] ? x1 : x0) + off[i]));
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        // partner vector: the same pairs of the other half (lane ^ G, same head)
        const uint32_t own[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
        uint32_t par[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) par[w] = rope_partner<GSH>(own[w], G);
        if (hl + static_cast<uint32_t>(i) * hps < heads) {
            u32x4r r;
            uint32_t* o = reinterpret_cast<uint32_t*>(&r);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                if constexpr (F16) {
                    // each product rounded once (the f16 operand widens inside
                    // the multiply), then the sum
                    const float y0 = mul_f16_half<0>(cs[2 * w], own[w]) + mul_f16_half<0>(sn[2 * w], par[w]);
                    const float y1 = mul_f16_half<1>(cs[2 * w + 1], own[w]) + mul_f16_half<1>(sn[2 * w + 1], par[w]);
                    o[w] = static_cast<uint32_t>(f2h(y0)) | (static_cast<uint32_t>(f2h(y1)) << 16);
                } else {
                    o[w] = __float_as_uint(__uint_as_float(own[w]) * cs[w] + __uint_as_float(par[w]) * sn[w]);
                }
            }
            __builtin_nontemporal_store(r, reinterpret_cast<u32x4r*>((sec[i] ? out1 : out0) + off[i]));
        }
    }
}

// Launches the token engine when its layout applies: 16-byte aligned
// operands, (d/2) a multiple of the vector width with a power-of-two number
// of vectors per head (2G <= 64), cos/sin rows on 16-byte boundaries, at
// most 8 head steps per lane, and at least 8192 (token, head) rows.  Returns
// false to fall back to the per-pair kernels.
template <bool F16>
bool launch_rope_half_token(hipStream_t stream, const void* x0, void* out0, uint32_t heads0, const void* x1,
                            void* out1, uint32_t heads1, const float* cosine, const float* sine, uint32_t tokens,
                            uint32_t head_dim, uint32_t rope_stride) {
    constexpr uint32_t V = F16 ? 8 : 4;
    const uint32_t half = head_dim / 2;
    if (half == 0 || half % V != 0 || rope_stride % 4 != 0 || tokens == 0) return false;
    const uint32_t G = half / V;
    if (G > 32 || (G & (G - 1)) != 0) return false;
    if (!aligned(x0, 16) || !aligned(out0, 16) || !aligned(cosine, 16) || !aligned(sine, 16) ||
        (heads1 != 0 && (!aligned(x1, 16) || !aligned(out1, 16))))
        return false;
    const uint32_t g_shift = static_cast<uint32_t>(__builtin_ctz(G));
    const uint32_t hps = 32u >> g_shift;
    const uint32_t heads = heads0 + heads1;
    if (heads == 0) return false;
    // small batches are latency-bound and measured faster on the per-pair
    // kernels (SmolLM2 shape, 128 tokens x 12 heads: 4.2 against 4.4 us)
    if (static_cast<uint64_t>(tokens) * heads < 8192) return false;
    const uint32_t ni = (heads + hps - 1) / hps;
    const dim3 grid((tokens + 3) / 4);
    const uint8_t* a0 = static_cast<const uint8_t*>(x0);
    const uint8_t* a1 = static_cast<const uint8_t*>(x1);
    uint8_t* b0 = static_cast<uint8_t*>(out0);
    uint8_t* b1 = static_cast<uint8_t*>(out1);
#define ATLAS_ROPE_TOKEN_CASE(N)                                                                                 \
    case N:                                                                                                      \
        if (g_shift == 2)                                                                                        \
            hipLaunchKernelGGL((rope_half_token_kernel<F16, N, 2>), grid, dim3(256), 0, stream, tokens, head_dim,   \
                               heads0, heads1, rope_stride, g_shift, a0, a1, cosine, sine, b0, b1);              \
        else if (g_shift == 3)                                                                                   \
            hipLaunchKernelGGL((rope_half_token_kernel<F16, N, 3>), grid, dim3(256), 0, stream, tokens, head_dim,   \
                               heads0, heads1, rope_stride, g_shift, a0, a1, cosine, sine, b0, b1);              \
        else                                                                                                     \
            hipLaunchKernelGGL((rope_half_token_kernel<F16, N, -1>), grid, dim3(256), 0, stream, tokens, head_dim, \
                               heads0, heads1, rope_stride, g_shift, a0, a1, cosine, sine, b0, b1);              \
        return true;
    switch (ni) {
        ATLAS_ROPE_TOKEN_CASE(1) ATLAS_ROPE_TOKEN_CASE(2) ATLAS_ROPE_TOKEN_CASE(3) ATLAS_ROPE_TOKEN_CASE(4)
        ATLAS_ROPE_TOKEN_CASE(5) ATLAS_ROPE_TOKEN_CASE(6) ATLAS_ROPE_TOKEN_CASE(7) ATLAS_ROPE_TOKEN_CASE(8)
        default: return false;
    }
#undef ATLAS_ROPE_TOKEN_CASE
}

hipError_t launch_rope_half_pair_f32(hipStream_t stream, const float* x0, float* out0, uint32_t heads0,
                                     const float* x1, float* out1, uint32_t heads1, const float* cosine,
                                     const float* sine, uint32_t tokens, uint32_t head_dim, uint32_t rope_stride) {
    if (launch_rope_half_token<false>(stream, x0, out0, heads0, x1, out1, heads1, cosine, sine, tokens, head_dim,
                                      rope_stride))
        return hipGetLastError();
    const uint32_t half = head_dim / 2;
    const bool vec = (half % 4) == 0 && (rope_stride % 4) == 0 && aligned(x0, 16) && aligned(out0, 16) &&
                     (heads1 == 0 || (aligned(x1, 16) && aligned(out1, 16))) && aligned(cosine, 16) &&
                     aligned(sine, 16);
    const uint32_t P = vec ? 4 : 1;
    const uint64_t threads = static_cast<uint64_t>(tokens) * (static_cast<uint64_t>(heads0) + heads1) * (half / P);
    const dim3 grid(static_cast<uint32_t>((threads + 255) / 256));
    if (vec)
        hipLaunchKernelGGL((rope_half_f32_kernel<4>), grid, dim3(256), 0, stream, tokens, head_dim, rope_stride,
                           heads0, heads1, x0, x1, cosine, sine, out0, out1);
    else
        hipLaunchKernelGGL((rope_half_f32_kernel<1>), grid, dim3(256), 0, stream, tokens, head_dim, rope_stride,
                           heads0, heads1, x0, x1, cosine, sine, out0, out1);
    return hipGetLastError();
}

hipError_t launch_rope_half_pair_f16(hipStream_t stream, const uint16_t* x0, uint16_t* out0, uint32_t heads0,
                                     const uint16_t* x1, uint16_t* out1, uint32_t heads1, const float* cosine,
                                     const float* sine, uint32_t tokens, uint32_t head_dim, uint32_t rope_stride) {
    if (launch_rope_half_token<true>(stream, x0, out0, heads0, x1, out1, heads1, cosine, sine, tokens, head_dim,
                                     rope_stride))
        return hipGetLastError();
    const uint32_t half = head_dim / 2;
    const bool vec = (half % 8) == 0 && (rope_stride % 4) == 0 && aligned(x0, 16) && aligned(out0, 16) &&
                     (heads1 == 0 || (aligned(x1, 16) && aligned(out1, 16))) && aligned(cosine, 16) &&
                     aligned(sine, 16);
    const uint32_t P = vec ? 8 : 1;
    const uint64_t threads = static_cast<uint64_t>(tokens) * (static_cast<uint64_t>(heads0) + heads1) * (half / P);
    const dim3 grid(static_cast<uint32_t>((threads + 255) / 256));
    if (vec)
        hipLaunchKernelGGL((rope_half_f16_kernel<8>), grid, dim3(256), 0, stream, tokens, head_dim, rope_stride,
                           heads0, heads1, x0, x1, cosine, sine, out0, out1);
    else
        hipLaunchKernelGGL((rope_half_f16_kernel<1>), grid, dim3(256), 0, stream, tokens, head_dim, rope_stride,
                           heads0, heads1, x0, x1, cosine, sine, out0, out1);
    return hipGetLastError();
}

hipError_t launch_rope_half_f32(hipStream_t stream, const float* x, const float* cosine, const float* sine,
                                float* out, uint32_t tokens, uint32_t heads, uint32_t head_dim,
                                uint32_t rope_stride) {
    return launch_rope_half_pair_f32(stream, x, out, heads, nullptr, nullptr, 0, cosine, sine, tokens, head_dim,
                                     rope_stride);
}

hipError_t launch_rope_half_f16(hipStream_t stream, const uint16_t* x, const float* cosine, const float* sine,
                                uint16_t* out, uint32_t tokens, uint32_t heads, uint32_t head_dim,
                                uint32_t rope_stride) {
    return launch_rope_half_pair_f16(stream, x, out, heads, nullptr, nullptr, 0, cosine, sine, tokens, head_dim,
                                     rope_stride);
}

hipError_t launch_rope_interleaved_f32(hipStream_t stream, const float* x, const float* cosine,
                                       const float* sine, float* out, uint32_t rows,
                                       uint32_t hidden) {
    const uint64_t threads = static_cast<uint64_t>(rows) * (hidden / 2);
    const dim3 grid(static_cast<uint32_t>((threads + 255) / 256));
    hipLaunchKernelGGL(rope_interleaved_kernel, grid, dim3(256), 0, stream, x, cosine, sine, out, rows,
                       hidden);
    return hipGetLastError();
}

}  // namespace atlas
