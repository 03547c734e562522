// norm_row_kernels.hip -- RMSNorm engines that give a row to a workgroup, for
// rows too wide for one wavefront's registers (hidden > 2048) and, in
// sequential order, for the row counts between a decode batch and a prefill.
//
// Semantics and the two reduction orders are norm_kernels.hip's.  A wavefront
// that holds a 4096-wide row alone keeps 192 registers of data and issues its
// 48 KB of loads and stores by itself; here NW wavefronts hold Q 16-byte
// columns each (column 64 (w + NW j) + l in lane l of wavefront w), so loads
// and stores spread over the CU and every input byte is read once.  Every row
// is read completely before any of its outputs is written, so in-place and
// aliased calls are safe.
#include "device_common.hpp"
#include "launch.hpp"
#include "norm_params.hpp"

namespace atlas {
namespace {

__device__ __forceinline__ f32x4 ldg_nt(const float* p) {
    return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
}
__device__ __forceinline__ void stg_nt(float* p, f32x4 v) {
    __builtin_nontemporal_store(v, reinterpret_cast<f32x4*>(p));
}

// The columns a thread holds of its row: x (for the add-norm x + residual once
// add() has run), the epilogue operand and the weight.
template <int NW, int Q, int MODE>
struct RowPart {
    static constexpr bool kOperand = MODE != kNormPlain;
    f32x4 x[Q], w[Q], e[kOperand ? Q : 1];

    static __device__ __forceinline__ uint32_t col(uint32_t tid, int j) { return tid + 64u * NW * j; }

    // x first: the sum waits for it alone while the operand and the weight
    // are still in flight
    __device__ __forceinline__ void load(const NormArgs& a, size_t base, uint32_t tid, uint32_t nv) {
        const float* operand = MODE == kNormAddScale ? a.out : a.residual;
#pragma unroll
        for (int j = 0; j < Q; ++j) x[j] = ldg_nt(a.x + base + 4 * min(col(tid, j), nv - 1));
        if (kOperand) {
#pragma unroll
            for (int j = 0; j < Q; ++j) e[j] = ldg_nt(operand + base + 4 * min(col(tid, j), nv - 1));
        }
#pragma unroll
        for (int j = 0; j < Q; ++j) w[j] = *reinterpret_cast<const f32x4*>(a.weight + 4 * min(col(tid, j), nv - 1));
        if (MODE == kNormAddNorm) {
#pragma unroll
            for (int j = 0; j < Q; ++j)
                x[j] = f32x4{x[j].x + e[j].x, x[j].y + e[j].y, x[j].z + e[j].z, x[j].w + e[j].w};
        }
    }

    __device__ __forceinline__ f32x4 square(int j, uint32_t tid, uint32_t nv) const {
        const f32x4 v = x[j];
        return col(tid, j) < nv ? f32x4{v.x * v.x, v.y * v.y, v.z * v.z, v.w * v.w} : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }

    __device__ __forceinline__ void finish(const NormArgs& a, size_t base, uint32_t tid, uint32_t nv, float inv,
                                           float scale) const {
#pragma unroll
        for (int j = 0; j < Q; ++j) {
            const uint32_t c = col(tid, j);
            if (c >= nv) continue;
            const f32x4 v = x[j], ww = w[j];
            const f32x4 n{v.x * inv * ww.x, v.y * inv * ww.y, v.z * inv * ww.z, v.w * inv * ww.w};
            const size_t at = base + 4 * c;
            if (MODE == kNormPlain) {
                stg_nt(a.out + at, n);
            } else if (MODE == kNormAddNorm) {
                stg_nt(a.residual_out + at, v);
                stg_nt(a.out + at, n);
            } else if (MODE == kNormResidual) {
                const f32x4 b = e[j];
                if (a.normalized) stg_nt(a.normalized + at, n);
                stg_nt(a.out + at, f32x4{b.x + n.x, b.y + n.y, b.z + n.z, b.w + n.w});
            } else {
                const f32x4 b = e[j];
                stg_nt(a.out + at,
                       f32x4{(b.x + n.x) * scale, (b.y + n.y) * scale, (b.z + n.z) * scale, (b.w + n.w) * scale});
            }
        }
    }
};

// Tree sum: a lane's columns, the wavefront (wave_sum_tree_f32), then the NW
// wavefronts' sums in order.
template <int NW, int Q, int MODE>
__global__ __launch_bounds__(64 * NW) void rms_row_tree_kernel(ATLAS_NORM_KPARAMS) {
    ATLAS_NORM_UNPACK;
    __shared__ float part[NW];
    const uint32_t tid = threadIdx.x, nv = a.hidden >> 2;
    const size_t base = static_cast<size_t>(blockIdx.x) * a.hidden;
    RowPart<NW, Q, MODE> r;
    r.load(a, base, tid, nv);
    const float scale = MODE == kNormAddScale ? *a.scale : 1.0f;
    float p = 0.0f;
#pragma unroll
    for (int j = 0; j < Q; ++j) {
        const f32x4 q = r.square(j, tid, nv);
        p = p + ((q.x + q.y) + (q.z + q.w));
    }
    p = wave_sum_tree_f32(p);
    if ((tid & 63u) == 0) part[tid >> 6] = p;
    __syncthreads();
    float s = part[0];
#pragma unroll
    for (int i = 1; i < NW; ++i) s = s + part[i];
    r.finish(a, base, tid, nv, inverse_rms(s, static_cast<float>(a.hidden), a.epsilon), scale);
}

// Sequential order, bit for bit, with the fold spread over the wavefronts:
//  1. every thread squares its columns into LDS; each 256-value block's sum in
//     any order goes beside them (an estimate: it only chooses binades);
//  2. wavefront 0 folds the head, the first 256 squares (head_fold_candidates),
//     while wavefront k >= 1 takes the k-th run of 64 S squares after it, lane
//     l the S consecutive ones from S l (S / 4 odd: the lanes' 16-byte reads
//     fall on distinct LDS banks), and computes chunk_scan for the binades that
//     the running sum can have inside its run by the estimates (at most three,
//     most often one or two);
//  3. the running sum goes from wavefront to wavefront, one barrier each; each
//     walks its run's events with the scans it has (chunk_walk) and falls back
//     to fold_chunk_exact_from outside them.
// Bound by that chain at few rows (an event costs ~250 cycles plus S adds, a
// row has 5 to 9) and by the scans' VALU work at many.
constexpr int kRowBinades = 3;

template <int NW, int Q, int S, int MODE>
__global__ __launch_bounds__(64 * NW) void rms_row_exact_kernel(ATLAS_NORM_KPARAMS) {
    ATLAS_NORM_UNPACK;
    constexpr uint32_t kBlocks = NW * Q;
    constexpr uint32_t kRunBlocks = S / 4;
    __shared__ __align__(16) f32x4 sq4[64 * kBlocks];
    __shared__ __align__(16) f32x4 head_pad[68];
    __shared__ float block_sum[kBlocks];
    __shared__ uint32_t running;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(tid >> 6));
    const uint32_t nv = a.hidden >> 2;
    const size_t base = static_cast<size_t>(blockIdx.x) * a.hidden;
    RowPart<NW, Q, MODE> r;
    r.load(a, base, tid, nv);
    const float scale = MODE == kNormAddScale ? *a.scale : 1.0f;
#pragma unroll
    for (int j = 0; j < Q; ++j) {
        const f32x4 q = r.square(j, tid, nv);
        const uint32_t block = wave + NW * j;
        sq4[64u * block + lane] = q;
        if (j == 0 && wave == 0) head_pad[lane + lane / 16] = q;
        const float t = wave_sum_any_order_f32((q.x + q.y) + (q.z + q.w));
        if (lane == 0) block_sum[block] = t;
    }
    __syncthreads();  // squares and block sums staged
    const uint32_t runs = ((nv + 63) / 64 + kRunBlocks - 2) / kRunBlocks;  // ceil((the row's blocks - 1) / kRunBlocks)
    float run[S];
    ChunkScan c[kRowBinades];
    uint32_t e0 = 0, binades = 0;
    if (wave == 0) {
        const float head = head_fold_candidates(head_pad, lane);
        if (lane == 0) running = __float_as_uint(head);
    } else if (wave <= runs) {
        const uint32_t first = kRunBlocks * (wave - 1) + 1;  // the run's first block
#pragma unroll
        for (int i = 0; i < S / 4; ++i) {
            const uint32_t at = 64u * first + kRunBlocks * lane + i;
            f32x4 q = sq4[min(at, 64u * kBlocks - 1)];
            if (kRunBlocks * (NW - 1) >= kBlocks && at >= 64u * kBlocks) q = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            run[4 * i] = q.x;
            run[4 * i + 1] = q.y;
            run[4 * i + 2] = q.z;
            run[4 * i + 3] = q.w;
        }
        const float mine = lane < kBlocks ? block_sum[lane] : 0.0f;
        const float before = wave_sum_any_order_f32(lane < first ? mine : 0.0f);
        const float after = wave_sum_any_order_f32(lane < first + kRunBlocks ? mine : 0.0f);
        // the in-order sum of <= 8192 squares is within 8192 * 2^-24 < 0.05 %
        // of the estimate, so these bound its exponent from both sides
        e0 = __float_as_uint(before * 0.999f) >> 23;
        const uint32_t e1 = __float_as_uint(after * 1.001f) >> 23;
        binades = min(e1 - e0 + 1u, static_cast<uint32_t>(kRowBinades));  // wave-uniform
#pragma unroll
        for (int b = 0; b < kRowBinades; ++b)
            if (static_cast<uint32_t>(b) < binades) c[b] = chunk_scan<S>(run, min(max(e0 + b, 27u), 251u));
    }
    for (uint32_t k = 1; k <= runs; ++k) {
        __syncthreads();  // the sum before run k is in `running`
        if (wave != k) continue;
        uint32_t sb = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(running));
        uint32_t l0 = 0;
#pragma unroll
        for (int b = 0; b < kRowBinades; ++b) {
            const uint32_t ex = e0 + b;
            if (static_cast<uint32_t>(b) < binades && l0 < 64 && (sb >> 23) == ex && ex >= 27 && ex <= 251)
                l0 = chunk_walk<S>(c[b], run, sb, l0, ex);
        }
        if (l0 < 64) sb = fold_chunk_exact_from<S>(run, sb, l0);
        if (lane == 0) running = sb;
    }
    __syncthreads();
    r.finish(a, base, tid, nv, inverse_rms(__uint_as_float(running), static_cast<float>(a.hidden), a.epsilon), scale);
}

template <int NW, int Q, int S, int MODE>
hipError_t launch_exact(hipStream_t s, const NormArgs& a) {
    static_assert(64 * NW * Q * 4 >= 256 + 256 && (S / 4) % 2 == 1, "the head and odd runs (LDS banks)");
    hipLaunchKernelGGL((rms_row_exact_kernel<NW, Q, S, MODE>), dim3(a.rows), dim3(64 * NW), 0, s,
                       ATLAS_NORM_KARGS(a, 1u, 0u));
    return hipGetLastError();
}

template <int NW, int Q, int MODE>
hipError_t launch_tree(hipStream_t s, const NormArgs& a) {
    hipLaunchKernelGGL((rms_row_tree_kernel<NW, Q, MODE>), dim3(a.rows), dim3(64 * NW), 0, s,
                       ATLAS_NORM_KARGS(a, 1u, 0u));
    return hipGetLastError();
}

// Shape of the exact engine: NW Q float4 columns hold the row, and the NW - 1
// runs of 64 S squares behind the 256 of the head end at or past it
// (256 + 64 S (NW - 1) values).  NW is a multiple of the four SIMDs (or half
// of them, two rows then share the SIMDs evenly): with six wavefronts a CU's
// rows queue on two of its SIMDs (1000 rows of 4096: 19.9 us with six, 11.3
// with four; 512 rows of 8192: 20.0 with twelve, 12.9 with eight).  Few rows
// want the work spread (a row's chain is all there is), many rows want few
// wavefronts per row (the scans of every run are VALU work).  Measured on
// MI355X, residual epilogue, us (graph of back-to-back launches):
//   hidden  rows    1      256    1000   4096   wavefront LDS engine before
//   2304            4.50   6.0    8.3    25.2   13.6 / 17.7 / 29.1 / 45.9
//   4096            5.2    7.5    11.2   37.0   23.2 / 34.1 / 49.6 / 139.8
//   8192            6.9    10.1   23.6   79.4   44.7 / 68.6 / 96.0 / 331.9
//   5120 <8,3,20>   5.8    8.1    17.5   57.5
//   5120 <4,5,28>   6.2    8.4    16.5   47.9
//   6144 <8,3,20>   5.9    8.7    19.2   63.3
//   6144 <4,6,36>   6.9    9.6    19.4   55.0
//   8192 <4,8,44>   8.3    11.8   26.2   86.1
// and at hidden <= 2048 between the decode and the prefill engines (RUN below,
// two rows per wavefront above; row-engine shapes <4,*,*> then <2,*,*>):
//   1536    rows    512: 5.95 RUN, 5.87    1000: 8.74 RUN, 6.92, 7.11
//                   1500: 11.4 RUN, 9.7, 8.2    2047: 14.5 RUN, 11.3, 9.3
template <int MODE>
hipError_t launch_exact_mode(hipStream_t s, const NormArgs& a) {
    const uint32_t h = a.hidden;
    if (h <= 2048 && a.rows >= 1024) {
        if (h <= 1536) return launch_exact<2, 3, 20, MODE>(s, a);
        return launch_exact<2, 4, 28, MODE>(s, a);
    }
    if (h <= 1024) return launch_exact<4, 1, 4, MODE>(s, a);
    if (h <= 2048) return launch_exact<4, 2, 12, MODE>(s, a);
    if (h <= 2560) return launch_exact<4, 3, 12, MODE>(s, a);
    if (h <= 3072) return launch_exact<4, 3, 20, MODE>(s, a);
    if (h <= 4096) return launch_exact<4, 4, 20, MODE>(s, a);
    if (h <= 6144 && a.rows < 768) return launch_exact<8, 3, 20, MODE>(s, a);
    if (h <= 5120) return launch_exact<4, 5, 28, MODE>(s, a);
    if (h <= 6144) return launch_exact<4, 6, 36, MODE>(s, a);
    return launch_exact<8, 4, 20, MODE>(s, a);
}

// [1000, 4096] plain 8.2 us (16.0 with one wavefront per row reading it
// twice), [4096, 4096] 24.3 (37.7); one row 2.5 (5.8).
template <int MODE>
hipError_t launch_tree_mode(hipStream_t s, const NormArgs& a) {
    const uint32_t h = a.hidden;
    if (h <= 3072) return launch_tree<4, 3, MODE>(s, a);
    if (h <= 4096) return launch_tree<4, 4, MODE>(s, a);
    if (h <= 6144) return launch_tree<8, 3, MODE>(s, a);
    return launch_tree<8, 4, MODE>(s, a);
}

template <int MODE>
hipError_t launch_mode(hipStream_t s, const NormArgs& a, bool tree) {
    return tree ? launch_tree_mode<MODE>(s, a) : launch_exact_mode<MODE>(s, a);
}

}  // namespace

bool rms_row_engine(const NormArgs& a, bool tree) {
    if (a.hidden > 2048) return a.hidden <= 8192;
    if (tree || a.hidden <= 256 || a.rows >= 2048) return false;
    return a.rows > (a.hidden > 1536 ? 256u : 512u);
}

hipError_t launch_rms_norm_row_f32(hipStream_t stream, NormMode mode, bool tree, const NormArgs& a) {
    switch (mode) {
        case kNormPlain: return launch_mode<kNormPlain>(stream, a, tree);
        case kNormResidual: return launch_mode<kNormResidual>(stream, a, tree);
        case kNormAddNorm: return launch_mode<kNormAddNorm>(stream, a, tree);
        case kNormAddScale: return launch_mode<kNormAddScale>(stream, a, tree);
    }
    return hipErrorInvalidValue;
}

}  // namespace atlas
