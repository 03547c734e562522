// logits_kernels.hip -- the decode tail of the Gemma executor: the final
// logit soft cap and the greedy argmax.
//
// Reference semantics (bisegni/atlas):
//   softcap_f32  crates/atlas-metal/src/kernels.metal:931-934
//                (v = cap * tanh(v / cap), in place; CPU form
//                gemma4_softcap_logits, crates/atlas-model/src/lib.rs:223-232)
//   argmax_f32   kernels.metal:2033-2066 (one 256-thread threadgroup: each
//                lane scans its stride with `value >= best`, then a tree keeps
//                the larger value or, on equal values, the larger index)
//   callers      gemma4_executor.rs:3673-3683 (prefill), :4678-4688 (decode)
//
// MI355X design.  The vocabulary row (262144 logits = 1 MiB) is split over
// many workgroups instead of one: each thread loads its float4s up front
// (nontemporal, every byte is touched once), caps them, stores them, and
// folds a 64-bit key per value,
//     key = (order(v) << 32) | index,
// where order() maps binary32 to an unsigned order (+0 and -0 share one
// code, NaN maps to 0 and so never wins).  The maximum key is the largest
// value and, among equal values, the largest index: exactly the reference's
// result, independent of how the row is split.  Keys reduce through the
// wavefront (shuffles) and the workgroup (LDS).  A row with one workgroup
// writes its index directly; otherwise every workgroup stores its key into
// its own slot of the context's workspace (plain stores, no atomics: many
// workgroups meeting on one word serialise at the memory-side atomic unit)
// and a second launch, one wavefront per row, reduces the row's slots.  The
// slots are overwritten by every launch, so the workspace needs no clearing.
#include "device_common.hpp"
#include "launch.hpp"

namespace atlas {
namespace {

constexpr int kLogitThreads = 256;

__device__ __forceinline__ uint64_t argmax_key(float v, uint32_t index) {
    uint32_t b = __float_as_uint(v);
    b = v == 0.0f ? 0u : b;  // -0 == +0 under the reference's comparisons
    const uint32_t ordered = (b & 0x80000000u) ? ~b : (b | 0x80000000u);  // -inf -> 0x007fffff
    const uint64_t key = (static_cast<uint64_t>(ordered) << 32) | index;
    return v != v ? 0ull : key;  // NaN never compares >= and is never taken
}

__device__ __forceinline__ uint64_t max_u64(uint64_t a, uint64_t b) { return a > b ? a : b; }

// The cap, and what a wavefront's plain values need of it: rcp = RN(1 / cap),
// formed on the host; 0 for a cap outside [2^-20, 2^20].
struct SoftCap {
    float cap, rcp;
};

SoftCap soft_cap(float cap) { return {cap, cap >= 0x1p-20f && cap <= 0x1p20f ? 1.0f / cap : 0.0f}; }

// cap * tanh(v / cap) for the values of one lane, with the bits of the IEEE
// steps (fdiv_rn, tanh_series_abs, tanh_exp_abs) throughout.  The series is
// evaluated for every value; the exponential only when some lane of the
// wavefront needs it (a wave-uniform branch), then selected per value.  Bound
// by this arithmetic where logits reach the exponential (|v| >= 0.625 cap), so
// both divisions are shorter ones where that is exact:
//  * v / cap in wavefronts whose |q0| = |v rcp| all lie in [2^-70, 2^60] --
//    ordinary logits; an exact zero, a mask's -inf or lowest float sends the
//    wavefront to the IEEE division: q0 is within 1.5 ulp of the quotient; q1 =
//    fma(v - q0 cap, rcp, q0) within half an ulp and a few 2^-22 of one, so
//    faithful; and q2 = fma(v - q1 cap, rcp, q1), with the residual exact (a
//    multiple of 2^-136; no operand comes near the subnormals) and rcp correctly
//    rounded, is the correctly rounded quotient (Markstein 1990).  Five
//    operations against the division's eleven;
//  * 2 / (e^{2a} + 1): tanh_exp_abs_with, enumerated equal over its whole
//    domain, for every wavefront.
// With wave_key below, soft cap + argmax of [256, 262144] at logits of standard
// deviation 8 and cap 30: 135 -> 95 us (the soft cap alone 119 -> 93, and with
// 2 % of the values at -inf 122 -> 103; 124 when such a wavefront took both
// long divisions behind the range test, which [256, 32000], a cache-resident
// batch, showed most: 16.6 -> 20.0, now 15.5); at deviation 1, where no value
// reaches the exponential, 93 both ways.
template <int N>
__device__ __forceinline__ void softcap_lanes(float (&v)[N], const SoftCap& k) {
    // the largest and smallest |q0|, not |v|: a product is never a signalling
    // NaN, which would take what max and min hold along with it
    float q0[N];
#pragma unroll
    for (int i = 0; i < N; ++i) q0[i] = v[i] * k.rcp;
    float hi = __builtin_fabsf(q0[0]), lo = hi;
#pragma unroll
    for (int i = 1; i < N; ++i) {
        hi = fmaxf(hi, __builtin_fabsf(q0[i]));
        lo = fminf(lo, __builtin_fabsf(q0[i]));
    }
    float a[N], r[N];
    // NaN among plain values: max and min skip it, every step propagates it
    // and the range test below leaves it to the series
    if (__builtin_amdgcn_ballot_w64(!(hi <= 0x1p60f && lo >= 0x1p-70f)) == 0) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float q1 = __builtin_fmaf(__builtin_fmaf(-q0[i], k.cap, v[i]), k.rcp, q0[i]);
            a[i] = __builtin_fabsf(__builtin_fmaf(__builtin_fmaf(-q1, k.cap, v[i]), k.rcp, q1));
        }
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) a[i] = __builtin_fabsf(fdiv_rn(v[i], k.cap));
    }
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = tanh_series_abs(a[i]);
    // q0 is within 1.5 ulp of the quotient: below 0.6249 none reaches 0.625
    if (__builtin_amdgcn_ballot_w64(hi >= 0.6249f || k.rcp == 0.0f) != 0) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float big = tanh_exp_abs_with<DivPositive>(a[i]);
            r[i] = a[i] >= 0.625f ? big : r[i];
        }
    }
    // cap > 0: the quotient's sign is v's
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = k.cap * __builtin_copysignf(r[i], v[i]);
}

// The wavefront's key over N float4 a lane, float4 u of lane l holding the
// values from index first + (u * kLogitThreads + l) * 4 on, or from `top` where
// that is less: the wavefront's maximum (NaN never raises it), then the last
// position that equals it, on the scalar unit from the comparisons' lane masks --
// two VALU operations a value where folding a 64-bit key per value takes ten.
// Wave-uniform.  RAW: values as loaded, which may be signalling NaNs; fmaxf loses
// what it holds beside one, so the first maximum is the propagating one, and
// where it is NaN a second takes the values quieted (quieting all of them:
// [128, 151936] 16.2 -> 16.8 us).
template <int N, bool RAW>
__device__ __forceinline__ uint64_t wave_key(const float (&x)[4 * N], uint32_t first, uint32_t top) {
    float m = x[0];
#pragma unroll
    for (int i = 1; i < 4 * N; ++i) m = RAW ? __builtin_elementwise_maximum(m, x[i]) : fmaxf(m, x[i]);
    if (RAW && __builtin_amdgcn_ballot_w64(m != m) != 0) {
        m = __builtin_canonicalizef(x[0]);
#pragma unroll
        for (int i = 1; i < 4 * N; ++i) m = fmaxf(m, __builtin_canonicalizef(x[i]));
    }
    m = wave_max_tree_f32(m);
    uint64_t key = 0;  // every value NaN
    bool open = true;
#pragma unroll
    for (int u = N - 1; u >= 0; --u) {
        uint64_t hit[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) hit[j] = __builtin_amdgcn_ballot_w64(x[4 * u + j] == m);
        const uint64_t any = (hit[0] | hit[1]) | (hit[2] | hit[3]);
        if (open && any != 0) {
            open = false;
            const uint32_t lane = 63u - static_cast<uint32_t>(__builtin_clzll(any));
            const uint32_t j = (hit[3] >> lane) & 1 ? 3u : ((hit[2] >> lane) & 1 ? 2u : ((hit[1] >> lane) & 1 ? 1u : 0u));
            key = argmax_key(m, min(first + (u * kLogitThreads + lane) * 4, top) + j);
        }
    }
    return key;
}

// Reduce a workgroup's key (the wavefront's already when UNIFORM) and publish
// it: the row's index when the row has one workgroup, otherwise the
// workgroup's slot of the workspace.
template <bool UNIFORM>
__device__ __forceinline__ void publish_key(uint64_t key, uint32_t row, uint64_t* slots, uint32_t* selected) {
    __shared__ uint64_t wave_keys[kLogitThreads / kWave];
    if (!UNIFORM)
        for (int off = kWave / 2; off > 0; off >>= 1) key = max_u64(key, __shfl_xor(key, off, kWave));
    const uint32_t lane = threadIdx.x % kWave;
    const uint32_t wave = threadIdx.x / kWave;
    if (lane == 0) wave_keys[wave] = key;
    __syncthreads();
    if (threadIdx.x != 0) return;
    key = wave_keys[0];
#pragma unroll
    for (int w = 1; w < kLogitThreads / kWave; ++w) key = max_u64(key, wave_keys[w]);
    if (gridDim.x == 1)
        selected[row] = static_cast<uint32_t>(key);
    else
        slots[static_cast<uint64_t>(row) * gridDim.x + blockIdx.x] = key;
}

// One wavefront per row: the maximum of the row's `per_row` slot keys.
__global__ __launch_bounds__(kLogitThreads) void argmax_finish_kernel(const uint64_t* slots, uint32_t per_row,
                                                                      uint32_t rows, uint32_t* selected) {
    const uint32_t row = blockIdx.x * (kLogitThreads / kWave) + threadIdx.x / kWave;
    if (row >= rows) return;  // whole wavefronts leave together
    const uint32_t lane = threadIdx.x % kWave;
    uint64_t key = 0;
    for (uint32_t i = lane; i < per_row; i += kWave) key = max_u64(key, slots[static_cast<uint64_t>(row) * per_row + i]);
    for (int off = kWave / 2; off > 0; off >>= 1) key = max_u64(key, __shfl_xor(key, off, kWave));
    if (lane == 0) selected[row] = static_cast<uint32_t>(key);
}

// Rows of `count` logits; blockIdx.y = row, blockIdx.x = slice of
// `per_block` values (a multiple of 1024 * U), walked in steps of 1024 * U.
// 16-byte accesses at any 4-byte alignment (count >= 4; a count that is not a
// multiple of 4 shifts every row); every load of a step is issued before its
// first value is processed.  A float4 that runs past the row is loaded from
// the row's last 4 values; the ones in front of its own position belong to
// the thread before it.  They are not stored, and the soft cap does not count
// them (in place, that thread may have stored already); the argmax alone counts
// them a second time, at their index.  [256, 50257] (one value a thread before):
// 39.3 -> 24.8 us, argmax of [256, 32001] 16.5 -> 9.4.
typedef f32x4 f32x4_row __attribute__((aligned(4)));

template <bool CAP, bool ARG, int U>
__global__ __launch_bounds__(kLogitThreads) void logits_vec_kernel(const float* in, float* out, uint32_t count,
                                                                   uint32_t per_block, float cap, float rcp,
                                                                   uint64_t* slots, uint32_t* selected) {
    const uint32_t row = blockIdx.y;
    const uint64_t base = static_cast<uint64_t>(row) * count;
    const uint32_t first = blockIdx.x * per_block;
    const uint32_t last = count - first < per_block ? count : first + per_block;
    const SoftCap k{cap, rcp};
    const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(threadIdx.x / kWave));
    uint64_t key = 0;
    for (uint32_t begin = first; begin < last; begin += kLogitThreads * 4 * U) {
        // short rows: no value of this step is this wavefront's (with U = 4 the
        // test costs more registers than it saves)
        if (U == 1 && begin + wave * (kWave * 4) >= last) break;
        float x[4 * U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = begin + (u * kLogitThreads + threadIdx.x) * 4;
            const uint32_t ic = min(i, count - 4);
            const f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4_row*>(in + base + ic));
            x[4 * u] = v.x;
            x[4 * u + 1] = v.y;
            x[4 * u + 2] = v.z;
            x[4 * u + 3] = v.w;
        }
        if (CAP) softcap_lanes(x, k);
        const bool whole = begin + kLogitThreads * 4 * U <= last;  // workgroup-uniform
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = begin + (u * kLogitThreads + threadIdx.x) * 4;
            if (CAP && out) {
                if (whole || i + 4 <= last) {
                    __builtin_nontemporal_store(f32x4{x[4 * u], x[4 * u + 1], x[4 * u + 2], x[4 * u + 3]},
                                                reinterpret_cast<f32x4_row*>(out + base + i));
                } else if (i < last) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (count - 4 + j >= i) out[base + count - 4 + j] = x[4 * u + j];
                }
            }
            if (CAP && ARG && !whole) {
                // position j of this float4 is index i + j: shift the tail's
                // values down and fill with NaN, which never wins
                const uint32_t skip = i + 4 <= last ? 0u : (i < last ? i + 4 - last : 4u);
                float y[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    y[j] = __builtin_nanf("");
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        if (j + s < 4) y[j] = skip == static_cast<uint32_t>(s) ? x[4 * u + j + s] : y[j];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) x[4 * u + j] = y[j];
            }
        }
        if (ARG) key = max_u64(key, wave_key<U, !CAP>(x, begin + wave * (kWave * 4), CAP ? 0xffffffffu : count - 4));
    }
    if (ARG) publish_key<true>(key, row, slots, selected);
}

// Rows of few values (launch_split): one value per thread per step.
template <bool CAP, bool ARG>
__global__ __launch_bounds__(kLogitThreads) void logits_scalar_kernel(const float* in, float* out, uint32_t count,
                                                                      uint32_t per_block, float cap, float rcp,
                                                                      uint64_t* slots, uint32_t* selected) {
    const uint32_t row = blockIdx.y;
    const uint64_t base = static_cast<uint64_t>(row) * count;
    const uint32_t begin = blockIdx.x * per_block;
    const uint32_t end = count - begin < per_block ? count : begin + per_block;
    const SoftCap k{cap, rcp};
    uint64_t key = 0;
    for (uint32_t i = begin + threadIdx.x; i < end; i += kLogitThreads) {
        float x[1] = {in[base + i]};
        if (CAP) softcap_lanes(x, k);
        if (CAP && out) out[base + i] = x[0];
        if (ARG) key = max_u64(key, argmax_key(x[0], i));
    }
    if (ARG) publish_key<false>(key, row, slots, selected);
}

// The grid of a soft cap / argmax over rows x count values: `blocks`
// workgroups per row, each covering `per_block` values.
struct RowSplit {
    bool vec, wide;
    uint32_t blocks, per_block;
};

RowSplit row_split(bool vec, bool wide, uint32_t rows, uint32_t count) {
    RowSplit r;
    r.vec = vec;
    // large batches: steps of 4096 values; a single row: 1024, for more
    // workgroups in flight.  At most kArgmaxSlotsPerRow workgroups per row:
    // longer rows give each workgroup several steps.
    r.wide = vec && wide && static_cast<uint64_t>(rows) * count >= (1u << 22);
    const uint32_t step = r.wide ? 4096u : 1024u;
    r.blocks = (count + step - 1) / step;
    r.per_block = step;
    if (r.blocks > kArgmaxSlotsPerRow) {
        r.per_block = ((count + kArgmaxSlotsPerRow - 1) / kArgmaxSlotsPerRow + step - 1) / step * step;
        r.blocks = (count + r.per_block - 1) / r.per_block;
    }
    return r;
}

bool aligned_rows(const float* in, const float* out, uint32_t count) {
    return count % 4 == 0 && (reinterpret_cast<uintptr_t>(in) & 15) == 0 &&
           (!out || (reinterpret_cast<uintptr_t>(out) & 15) == 0);
}

// The split that the no-allocation entry point's limit is stated in: rows
// that are not a multiple of 4 values, or not 16-byte aligned, count their
// workgroups in steps of 1024 values at any batch size.  The launch itself
// needs at most as many.
RowSplit limit_split(const float* in, const float* out, uint32_t rows, uint32_t count) {
    const bool aligned = aligned_rows(in, out, count);
    return row_split(aligned, aligned, rows, count);
}

// The split of a launch.  Aligned rows take float4 steps from 4 values on, and
// so does an argmax of any row.  The soft cap of unaligned rows computes every
// value that its float4 repeat: short rows go one value a thread, and rows that
// would fill less than 0.6 of their wide steps take narrow ones.  Soft cap +
// argmax of [4000, n], us, one value a thread / narrow / wide:
//   n = 5     5.5 / 6.4 / -         129   6.9 / 7.5 / -       ([1000, 385] 4.5 / 4.9)
//   n = 513   10.7 / 8.8 / -        1537  27 / 18.5 / 22.8    (masked 27 / 19.3 / 29)
//   n = 4097  52 / 36 / 42 (masked 51 / 36 / 50)
//   n = 8193  96 / 65 / 58 (masked 93 / 64 / 70)              12001  135 / 88 / 76
template <bool CAP>
RowSplit launch_split(const float* in, const float* out, uint32_t rows, uint32_t count) {
    const bool loose = CAP && !aligned_rows(in, out, count);
    const uint64_t wide_steps = (static_cast<uint64_t>(count) + 4095) / 4096 * 4096;
    return row_split(count >= (loose ? 512u : 4u), !loose || 5ull * count >= 3 * wide_steps, rows, count);
}

// Rows one launch can cover with `slot_count` workspace slots (a row split
// over one workgroup writes its result directly and needs none).
uint32_t row_launch_rows(uint32_t blocks, uint32_t slot_count) {
    return blocks == 1 ? 65535u : slot_count / blocks;
}

template <bool CAP, bool ARG>
hipError_t launch_rows(hipStream_t stream, const float* in, float* out, uint32_t* selected, uint32_t rows,
                       uint32_t count, float cap, uint64_t* slots, uint32_t slot_count) {
    const SoftCap k = soft_cap(cap);
    const RowSplit split = launch_split<CAP>(in, out, rows, count);
    const bool vec = split.vec, wide = split.wide;
    const uint32_t blocks = split.blocks, per_block = split.per_block;
    const uint32_t rows_per_launch = row_launch_rows(blocks, slot_count);
    for (uint32_t r0 = 0; r0 < rows; r0 += rows_per_launch) {
        const uint32_t n = rows - r0 < rows_per_launch ? rows - r0 : rows_per_launch;
        const dim3 grid(blocks, n);
        const float* rin = in + static_cast<uint64_t>(r0) * count;
        float* rout = out ? out + static_cast<uint64_t>(r0) * count : nullptr;
        uint32_t* rsel = ARG ? selected + r0 : nullptr;
        if (vec && wide)
            hipLaunchKernelGGL((logits_vec_kernel<CAP, ARG, 4>), grid, dim3(kLogitThreads), 0, stream, rin, rout,
                               count, per_block, k.cap, k.rcp, slots, rsel);
        else if (vec)
            hipLaunchKernelGGL((logits_vec_kernel<CAP, ARG, 1>), grid, dim3(kLogitThreads), 0, stream, rin, rout,
                               count, per_block, k.cap, k.rcp, slots, rsel);
        else
            hipLaunchKernelGGL((logits_scalar_kernel<CAP, ARG>), grid, dim3(kLogitThreads), 0, stream, rin, rout,
                               count, per_block, k.cap, k.rcp, slots, rsel);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        if (ARG && blocks > 1) {
            const uint32_t waves = kLogitThreads / kWave;
            hipLaunchKernelGGL(argmax_finish_kernel, dim3((n + waves - 1) / waves), dim3(kLogitThreads), 0, stream,
                               slots, blocks, n, rsel);
            e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

// Soft cap of a flat array: grid-stride float4 body plus a scalar tail.
__global__ __launch_bounds__(kLogitThreads) void softcap_vec_kernel(const float* in, float* out, uint64_t n4,
                                                                    float cap, float rcp) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    const SoftCap k{cap, rcp};
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n4; i += stride) {
        const f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(in) + i);
        float x[4] = {v.x, v.y, v.z, v.w};
        softcap_lanes(x, k);
        __builtin_nontemporal_store(f32x4{x[0], x[1], x[2], x[3]}, reinterpret_cast<f32x4*>(out) + i);
    }
}

__global__ __launch_bounds__(kLogitThreads) void softcap_scalar_kernel(const float* in, float* out, uint64_t begin,
                                                                       uint64_t n, float cap, float rcp) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    const SoftCap k{cap, rcp};
    for (uint64_t i = begin + static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
        float x[1] = {in[i]};
        softcap_lanes(x, k);
        out[i] = x[0];
    }
}

uint32_t grid_for(uint64_t items) {
    const uint64_t blocks = (items + kLogitThreads - 1) / kLogitThreads;
    return static_cast<uint32_t>(blocks < 8192 ? (blocks ? blocks : 1) : 8192);
}

}  // namespace

size_t argmax_workspace_bytes() { return kArgmaxSlots * sizeof(uint64_t); }

hipError_t launch_logits_f32(hipStream_t stream, const float* logits, float* capped, uint32_t* selected,
                             uint32_t rows, uint32_t count, float cap, void* workspace, uint32_t slot_count) {
    uint64_t* slots = static_cast<uint64_t*>(workspace);
    const bool do_cap = cap > 0.0f;
    if (do_cap && selected)
        return launch_rows<true, true>(stream, logits, capped, selected, rows, count, cap, slots, slot_count);
    if (selected)
        return launch_rows<false, true>(stream, logits, nullptr, selected, rows, count, cap, slots, slot_count);
    return launch_rows<true, false>(stream, logits, capped, nullptr, rows, count, cap, slots, slot_count);
}

uint32_t logits_launches(const float* logits, const float* capped, uint32_t rows, uint32_t count,
                         uint32_t slot_count) {
    const RowSplit split = limit_split(logits, capped, rows, count);
    const uint32_t per = row_launch_rows(split.blocks, slot_count);
    return per == 0 ? 0u : (rows + per - 1) / per;
}

uint32_t logits_row_blocks(const float* logits, const float* capped, uint32_t rows, uint32_t count) {
    return limit_split(logits, capped, rows, count).blocks;
}

// ---------------------------------------------------------------------------
// Scratch of the no-allocation soft cap + argmax entry point: a file-scope
// device array, one per GPU for the life of the process.  Host code never
// passes the symbol itself to a kernel (on the host it is only a stand-in);
// argmax_scratch_address resolves this device's copy once, with the device
// current, and callers pass that address.  Every slot a call reads is
// written by the same call first, so the array needs no clearing; calls
// that overlap on one GPU share it and race.
// ---------------------------------------------------------------------------
static __device__ __align__(256) uint64_t scratch[kArgmaxScratchSlots];

hipError_t argmax_scratch_address(void** ptr) {
    return hipGetSymbolAddress(ptr, HIP_SYMBOL(scratch));
}

hipError_t launch_softcap_f32(hipStream_t stream, const float* in, float* out, uint64_t n, float cap) {
    const bool vec = (reinterpret_cast<uintptr_t>(in) & 15) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    const uint64_t n4 = vec ? n / 4 : 0;
    const SoftCap k = soft_cap(cap);
    if (n4) {
        hipLaunchKernelGGL(softcap_vec_kernel, dim3(grid_for(n4)), dim3(kLogitThreads), 0, stream, in, out, n4, k.cap,
                           k.rcp);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    if (n4 * 4 < n) {
        hipLaunchKernelGGL(softcap_scalar_kernel, dim3(grid_for(n - n4 * 4)), dim3(kLogitThreads), 0, stream, in, out,
                           n4 * 4, n, k.cap, k.rcp);
        return hipGetLastError();
    }
    return hipSuccess;
}

}  // namespace atlas
