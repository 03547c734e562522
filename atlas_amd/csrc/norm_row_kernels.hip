// norm_row_kernels.hip -- RMSNorm engines that give a row to a workgroup, for
// rows too wide for one wavefront's registers (hidden > 2048) and, in
// sequential order, for narrower rows below the prefill's row counts.
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

// Sequential order, bit for bit, from segments of 64 squares folded side by
// side.  Inside a binade a running sum is an integer count of its ulps, and
// adding a non-negative value raises it by a whole number of ulps that depends
// on the sum only through its parity (a tie rounds to even).  So a segment
// that stays in the binade raises every even sum by one amount and every odd
// sum by another, and a run of such segments is a function of the parity at
// its start.
//  1. Every thread squares its columns into LDS; each segment's sum in any
//     order goes beside them, and every wavefront scans those into estimates
//     of the segments' starts.
//  2. Wavefront 0 folds the head, the first 256 squares (head_fold_candidates).
//     The next PW wavefronts fold every later segment from an even and an odd
//     start at its estimate, a lane each, 32 segments a pass, and compose the
//     segments between crossings into runs by a wave scan.  The rest take the
//     segments that may cross a power of two by the estimates (with a margin of
//     64 ulps: a segment's in-order sum is within 32 of any other order's):
//     windows of consecutive starts around the estimate, a lane each.
//  3. Each window's lane goes on from its fold through the run behind it (one
//     integer add a group of 32 segments, the binade checked at both ends), and
//     wavefront 0 from the head through the first run.
//  4. Every wavefront follows the exact sum from window to window, one readlane
//     each: about log2(hidden / 256) of them.
// What the estimates missed -- a start outside its window, more crossings than
// windows, a binade they put elsewhere -- is folded in order from the exact sum
// (wavefront 0), and the way goes on with the next window.  Every step is the
// in-order fold's own adds or provably equals them, so the result is its bit
// pattern.
//
// A sum strays from its estimate by the rounding since the last power of two,
// about 0.3 sqrt(values) ulps: 32 starts hold it to 1000 values, 64 to the
// widest row.  With few rows the time is one chain: load, 64 adds behind 16
// LDS reads, scan, runs, three barriers.  One row of 1536 (residual) 2.9 us,
// against 3.4 with one wavefront folding whole chunks under helpers' scans
// (and 2.2 for the tree sum); 4096: 3.4 (5.2 with runs of 4 to 36 float4 a
// lane); 8192: 4.7 (6.9); [256, 1536] 4.1 (4.6).  Following the sum step by
// step in wavefront 0, with the runs and windows published as they are: 3.4 at
// 1536, 4.1 at 4096.
constexpr uint32_t kSegMargin = 64;
constexpr uint32_t kNoParity = 0xffffffffu;  // the segment left its binade
constexpr uint32_t kNoSum = 0xffffffffu;     // no exact sum from this start
constexpr uint32_t kGroup = 32;              // segments of one parity pass, two lanes each

// Sum over each 16-lane row, in every lane (any order).
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_f32<0xb1, 0xf, false>(v);
    v += dpp_f32<0x4e, 0xf, false>(v);
    v += dpp_f32<0x141, 0xf, false>(v);
    return v + dpp_f32<0x140, 0xf, false>(v);
}

// Ulps that a run of segments adds to an even (e) and to an odd (o) sum; f
// marks that the run begins behind a crossing.
struct ParityRun {
    uint32_t e, o, f;
};

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void compose_step(ParityRun& b) {
    const uint32_t ae = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(b.e), CTRL, ROW_MASK, 0xf, false));
    const uint32_t ao = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(b.o), CTRL, ROW_MASK, 0xf, false));
    const uint32_t af = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(b.f), CTRL, ROW_MASK, 0xf, false));
    const uint32_t e = ae + ((ae & 1u) ? b.o : b.e), o = ao + ((ao & 1u) ? b.e : b.o);
    b.e = b.f ? b.e : e;
    b.o = b.f ? b.o : o;
    b.f |= af;
}

__device__ __forceinline__ float fold_regs_16(const f32x4 (&v)[16], float s) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        s = s + v[i].x;
        s = s + v[i].y;
        s = s + v[i].z;
        s = s + v[i].w;
    }
    return s;
}

template <int NW, int Q, int PW, int HALF, int MODE>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 4 && Q == 4 ? 4 : 1)))
void rms_row_exact_kernel(ATLAS_NORM_KPARAMS) {
    ATLAS_NORM_UNPACK;
    constexpr uint32_t kSegs = 4 * NW * Q;  // segments of 16 float4 that the threads hold
    constexpr int G = (kSegs + 63) / 64;    // registers of one segment per lane
    constexpr int kCross = NW - 1 - PW;     // wavefronts with windows
    // windows: two of 32 starts in each of the first HALF such wavefronts, one of 64 in each other
    constexpr uint32_t kHalves = 2 * HALF, kWindows = kCross + HALF;
    static_assert(PW >= 1 && HALF >= 0 && HALF <= kCross && kCross >= 1 && G <= 2, "wavefront roles");
    __shared__ __align__(16) f32x4 sq4[17 * kSegs];  // float4 c at c + c / 16: 16 lanes on distinct banks
    __shared__ float seg_sum[64 * G];
    __shared__ __align__(16) u32x4_t runs[kSegs];  // by a run's last segment: ulps from an even, an odd sum; binade
    __shared__ uint32_t cand[64 * kCross];       // the sum behind a crossing and its run, by the start in the window
    __shared__ uint32_t window[64];              // a window's first start
    __shared__ uint32_t first_sum, total;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(tid >> 6));
    const uint32_t nv = a.hidden >> 2, nseg = (nv + 15) / 16;
    const size_t base = static_cast<size_t>(blockIdx.x) * a.hidden;
    RowPart<NW, Q, MODE> r;
    r.load(a, base, tid, nv);
    const float scale = MODE == kNormAddScale ? *a.scale : 1.0f;
#pragma unroll
    for (int j = 0; j < Q; ++j) {
        const f32x4 q = r.square(j, tid, nv);
        const uint32_t c = r.col(tid, j);
        sq4[c + c / 16] = q;
        const float t = row16_sum((q.x + q.y) + (q.z + q.w));
        if (lane % 16 == 0) seg_sum[c / 16] = t;
    }
    __syncthreads();  // squares and segment sums staged

    float own[G];
#pragma unroll
    for (int g = 0; g < G; ++g) own[g] = lane + 64u * g < kSegs ? seg_sum[lane + 64u * g] : 0.0f;
    auto load_segment = [&](f32x4 (&v)[16], uint32_t k) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = sq4[17 * k + i];
    };
    // est[g]: the estimated start of segment lane + 64 g; cross: the segments
    // that may leave its binade
    uint32_t est[G];
    uint64_t cross[G];
    auto scan_estimates = [&] {
        float before = 0.0f;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const uint32_t k = lane + 64u * g;
            const float incl = before + wave_inclusive_scan_f32(own[g]);
            const float excl = __int_as_float(
                __builtin_amdgcn_update_dpp(__float_as_int(before), __float_as_int(incl), 0x138, 0xf, 0xf, false));  // wave_shr:1
            before = readlane_f32(incl, 63);
            est[g] = __float_as_uint(excl);
            const bool in = k >= 4 && k < nseg;
            cross[g] = __builtin_amdgcn_ballot_w64(
                in && (max(est[g], kSegMargin) - kSegMargin) >> 23 != (__float_as_uint(incl) + kSegMargin) >> 23);
        }
    };
    auto estimate = [&](uint32_t k) {  // any segment's, per lane
        uint32_t e = static_cast<uint32_t>(__shfl(static_cast<int>(est[0]), static_cast<int>(k & 63u), kWave));
        if (G > 1) {
            const uint32_t w = static_cast<uint32_t>(__shfl(static_cast<int>(est[G - 1]), static_cast<int>(k & 63u), kWave));
            e = k >= 64 ? w : e;
        }
        return e;
    };

    // takes the lowest of the segments that may cross; nseg when there is none
    auto take_crossing = [&](uint64_t& left0, uint64_t& left1) {
        const uint32_t p = left0 ? static_cast<uint32_t>(__builtin_ctzll(left0))
                                 : (left1 ? 64u + static_cast<uint32_t>(__builtin_ctzll(left1)) : nseg);
        const uint64_t low0 = left0 & (left0 - 1), low1 = left1 & (left1 - 1);
        left1 = left0 ? left1 : low1;
        left0 = left0 ? low0 : 0;
        return p;
    };
    // the sum behind the runs from segment pos to the crossing p, from s at pos
    auto through_runs = [&](uint32_t s, uint32_t pos, uint32_t p, bool& ok) {
#pragma unroll
        for (uint32_t k0 = 0; k0 < kSegs; k0 += kGroup) {
            const uint32_t end = min(p, k0 + kGroup);
            const bool in = max(pos, k0) < end;
            const u32x4_t run = runs[in ? end - 1 : 0];
            const uint32_t to = s + ((s & 1u) ? run.y : run.x);
            ok = ok && (!in || (((s ^ run.z) | (to ^ run.z)) >> 23) == 0);
            s = in ? to : s;
        }
        return s;
    };

    uint32_t sum = 0;                // wavefront 0: the bits of the sum behind the head; a window lane's behind its segment
    uint32_t pos = 4, upto = nseg;  // the run that follows
    if (wave == 0) {
        const uint32_t head_seg = lane == 0 ? 0u : (lane - 1) / 21 + 1;
        const uint32_t j = lane == 0 ? 0u : (lane - 1) % 21;
        f32x4 v[16];
        load_segment(v, head_seg);  // on its way while the estimates are scanned
        scan_estimates();
        // the head, as head_fold_candidates: segment 0 from 0, each of the
        // next three from the 21 floats around its estimate, then selected
        uint32_t e[4];
#pragma unroll
        for (uint32_t k = 1; k < 4; ++k) e[k] = readlane_u32(est[0], k) - 10u;
        const uint32_t start = head_seg == 0 ? 0u : (head_seg == 1 ? e[1] : (head_seg == 2 ? e[2] : e[3])) + j;
        const float res = fold_regs_16(v, __uint_as_float(start));
        sum = readlane_u32(__float_as_uint(res), 0);
#pragma unroll
        for (uint32_t k = 1; k < 4; ++k) {
            const uint32_t at = sum - e[k];
            if (__builtin_expect(at < 21, 1))
                sum = readlane_u32(__float_as_uint(res), 21 * k - 20 + at);
            else
                sum = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(
                    __float_as_uint(fold_lds_16(sq4 + 17 * k, __uint_as_float(sum)))));
        }
        uint64_t left0 = cross[0], left1 = G > 1 ? cross[G - 1] : 0;
        upto = take_crossing(left0, left1);
    } else if (wave <= PW) {
        f32x4 v[16];
        load_segment(v, min(kGroup * (wave - 1) + (lane >> 1), nseg - 1));
        scan_estimates();
        for (uint32_t k0 = kGroup * (wave - 1); k0 < nseg; k0 += kGroup * PW) {
            const uint32_t k = k0 + (lane >> 1), kc = min(k, nseg - 1);
            if (k0 >= kGroup * PW) load_segment(v, kc);  // a later pass
            const uint32_t start = (estimate(kc) & ~1u) | (lane & 1u);
            const uint32_t end = __float_as_uint(fold_regs_16(v, __uint_as_float(start)));
            const bool crosses = ((k < 64 ? cross[0] : cross[G - 1]) >> (k & 63u)) & 1;
            const uint32_t mine = (start >> 23) == (end >> 23) ? end - start : kNoParity;
            const uint32_t other = static_cast<uint32_t>(
                __builtin_amdgcn_update_dpp(0, static_cast<int>(mine), 0xb1, 0xf, 0xf, false));  // the other parity's
            const bool lost = mine == kNoParity || other == kNoParity;
            ParityRun run{lane & 1u ? other : mine, lane & 1u ? mine : other, 0u};
            if (crosses || lost || k < 4) run = ParityRun{0u, 0u, 1u};  // (the head is not part of a run)
            compose_step<0x112, 0xf>(run);  // row_shr:2, 4, 8: a segment has two lanes
            compose_step<0x114, 0xf>(run);
            compose_step<0x118, 0xf>(run);
            compose_step<0x142, 0xa>(run);
            compose_step<0x143, 0xc>(run);
            // (a lost one means a wrong estimate: no run of this pass holds)
            const bool wrong = __builtin_amdgcn_ballot_w64(lost && !crosses && k >= 4 && k < nseg) != 0;
            const uint32_t binade = (start >> 23) ^ (wrong ? 0x80u : 0u);
            if (k < nseg && !(lane & 1u)) runs[k] = u32x4_t{run.e, run.o, binade << 23, 0u};
        }
    } else {
        scan_estimates();
        // this wavefront's windows: crossing number first + i in lanes CW i ..
        const uint32_t part = wave - 1 - PW;
        const bool half = part < HALF;
        const uint32_t first = half ? 2 * part : part + HALF, width = half ? 32u : 64u;
        uint64_t left0 = cross[0], left1 = G > 1 ? cross[G - 1] : 0;
        for (uint32_t i = 0; i < first; ++i) take_crossing(left0, left1);
        const uint32_t p0 = take_crossing(left0, left1), p1 = take_crossing(left0, left1), p2 = take_crossing(left0, left1);
        const bool second = half && lane >= 32;
        const uint32_t k = min(second ? p1 : p0, nseg - 1);  // (the last one: a window that no crossing needs)
        upto = second ? p2 : p1;
        pos = k + 1;
        const uint32_t from = estimate(k) - width / 2;
        if (lane % width == 0) window[first + (second ? 1u : 0u)] = from;
        sum = __float_as_uint(fold_lds_16(sq4 + 17 * k, __uint_as_float(from + lane % width)));
    }
    __syncthreads();  // every run published
    if (wave == 0 || wave > PW) {
        bool ok = true;
        const uint32_t to = through_runs(sum, pos, upto, ok);
        uint32_t* at = wave == 0 ? &first_sum : cand + 64 * (wave - 1 - PW) + lane;
        if (wave != 0 || lane == 0) *at = ok ? to : kNoSum;
    }
    __syncthreads();  // every sum behind a crossing and its run published
    // every wavefront goes from crossing to crossing
    uint32_t res[kCross];
#pragma unroll
    for (int i = 0; i < kCross; ++i) res[i] = cand[64 * i + lane];
    const uint32_t windows = window[lane];
    const uint32_t crossings = __builtin_popcountll(cross[0]) + (G > 1 ? __builtin_popcountll(cross[G - 1]) : 0);
    uint32_t sb = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(first_sum)), passed = 0;
    bool on = sb != kNoSum;
    const bool started = on;
#pragma unroll
    for (uint32_t w = 0; w < kWindows; ++w) {
        const uint32_t width = w < kHalves ? 32 : 64;
        const uint32_t at = sb - readlane_u32(windows, w);
        const uint32_t to = w < kHalves ? readlane_u32(res[w / 2], w % 2 * 32 + at % 32) : readlane_u32(res[w - HALF], at % 64);
        on = on && w < crossings && at < width && to != kNoSum;
        sb = on ? to : sb;
        passed += on;
    }
    if (__builtin_expect(!started || passed < crossings, 0)) {
        // a start outside its window, or a run that is not the binade's: folded
        // in order from the exact sum
        if (wave == 0) {
            uint64_t left0 = cross[0], left1 = G > 1 ? cross[G - 1] : 0;
            uint32_t p = take_crossing(left0, left1), w = 0;  // the next crossing, its number
            for (; w < passed; ++w) p = take_crossing(left0, left1);
            uint32_t s = started ? sb : sum, k = started ? p : 4;
            while (k < nseg) {
                const uint32_t stop = k < p ? p : k + 1;  // the run before the crossing p, or p itself
                uint32_t to, behind = stop;
                bool ok = true;
                if (k < p) {
                    to = through_runs(s, k, p, ok);
                } else {
                    p = take_crossing(left0, left1);
                    const uint32_t v = min(w, kWindows - 1), width = v < kHalves ? 32 : 64;
                    const uint32_t at = s - window[v];
                    to = cand[(v < kHalves ? 32 * v : 64 * (v - HALF)) + at % width];
                    ok = w < kWindows && at < width && to != kNoSum;
                    behind = p;
                    ++w;
                }
                if (ok) {
                    s = to;
                    k = behind;
                }
                for (; !ok && k < stop; ++k) s = __float_as_uint(fold_lds_16(sq4 + 17 * k, __uint_as_float(s)));
            }
        if (lane == 0) total = s;
        }
        __syncthreads();
        sb = total;
    }
    r.finish(a, base, tid, nv, inverse_rms(__uint_as_float(sb), static_cast<float>(a.hidden), a.epsilon), scale);
}

template <int NW, int Q, int PW, int HALF, int MODE>
hipError_t launch_exact(hipStream_t s, const NormArgs& a) {
    hipLaunchKernelGGL((rms_row_exact_kernel<NW, Q, PW, HALF, MODE>), dim3(a.rows), dim3(64 * NW), 0, s,
                       ATLAS_NORM_KARGS(a, 1u, 0u));
    return hipGetLastError();
}

template <int NW, int Q, int MODE>
hipError_t launch_tree(hipStream_t s, const NormArgs& a) {
    hipLaunchKernelGGL((rms_row_tree_kernel<NW, Q, MODE>), dim3(a.rows), dim3(64 * NW), 0, s,
                       ATLAS_NORM_KARGS(a, 1u, 0u));
    return hipGetLastError();
}

// Wavefronts and columns by width, and by rows: up to two workgroups a CU the
// eight-wavefront shapes win (a thread holds less, and every window has 64
// starts), past that the four-wavefront ones, which fit more often.  Residual
// epilogue, us, eight / four wavefronts: [512, 1536] 4.9 / 4.9, [700, 1536]
// 6.9 / 5.4; [512, 2048] 5.2 / 5.4, [700, 2048] 7.2 / 6.0; [512, 3072] 6.2 / 7.0,
// [700, 3072] 8.8 / 7.8; [512, 4096] 7.0 / 8.1, [700, 4096] 9.7 / 9.2;
// [256, 8192] 8.7 / 10.6, [512, 8192] 15.5 / 13.1 (one workgroup a CU there).
// To 1024 one column a thread leaves nothing to split: [1, 1024] 2.9 / 2.7.
template <int MODE>
hipError_t launch_exact_mode(hipStream_t s, const NormArgs& a) {
    const uint32_t h = a.hidden;
    const bool few = a.rows <= 512;
    if (h <= 1024) return launch_exact<4, 1, 1, 2, MODE>(s, a);
    if (h <= 2048) return few ? launch_exact<8, 1, 1, 0, MODE>(s, a) : launch_exact<4, 2, 1, 1, MODE>(s, a);
    if (h <= 4096 && few) return launch_exact<8, 2, 2, 0, MODE>(s, a);
    if (h <= 3072) return launch_exact<4, 3, 1, 2, MODE>(s, a);
    if (h <= 4096) return launch_exact<4, 4, 1, 2, MODE>(s, a);
    if (h <= 6144) return launch_exact<8, 3, 3, 1, MODE>(s, a);
    if (a.rows <= 256) return launch_exact<8, 4, 2, 1, MODE>(s, a);
    return launch_exact<4, 8, 1, 2, MODE>(s, a);
}

// [1000, 4096] plain 7.4 us (16.3 with one wavefront per row reading it
// twice), [4096, 4096] 24.0 (36.9); one row 2.5 (5.8).
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

// Sequential order, us by the per-wavefront engine (with its helpers) / by
// this one, residual epilogue:
//   rows       1            64           256          512          1000         2047
//   516 wide   3.06 / 3.12  4.08 / 4.04  4.29 / 4.20  4.56 / 4.57  6.56 / 5.33  10.5 / 7.94
//   576        3.10 / 3.10  3.85 / 3.88  4.05 / 3.92  4.46 / 4.22  6.23 / 4.88  10.0 / 7.47
//   768        3.16 / 3.11  3.97 / 3.81  4.19 / 4.04  4.50 / 4.44  6.52 / 5.32  10.4 / 7.86
//   1000       3.66 / 3.30  4.44 / 4.08  4.74 / 4.44  5.12 / 4.95  7.37 / 5.76  11.3 / 8.45
// To 512 wide it takes over as rows queue ([700, 512] 3.9 / 4.0, [1000, 512]
// 5.27 / 4.82, [2047, 512] 7.58 / 7.22, [1000, 384] 5.02 / 4.70, [2047, 384]
// 7.25 / 7.12), below 384 it does not pay ([1700, 260] 6.55 / 6.91, [1700, 320]
// 6.29 / 6.55).  From 2048 rows up to 2048 wide two rows a wavefront keep more
// loads in flight: [2048, 576] 6.7 (7.5 by this one at 2047), [2048, 1536]
// 9.8 / 9.9, [4096, 1536] 13.6 / 16.8 (one row a wavefront: [2047, 1536] 14.5 / 9.9).  Past 2048 wide
// there is no other engine to 8192.
bool rms_row_engine(const NormArgs& a, bool tree) {
    if (a.hidden > 2048) return a.hidden <= 8192;
    if (tree || a.rows >= 2048) return false;
    return a.hidden > 512 || (a.hidden >= 384 && a.rows > 800);
}

hipError_t launch_rms_norm_row_f32(hipStream_t stream, NormMode mode, bool tree, const NormArgs& args) {
    // a launch's threads are counted in 32 bits (past that only the remainder
    // runs, without an error), and a row here has up to 512
    constexpr uint32_t kRowsPerLaunch = 0xffffffffu / 512;
    hipError_t e = hipErrorInvalidValue;
    for (uint64_t r0 = 0; r0 < args.rows; r0 += kRowsPerLaunch) {
        const uint64_t at = r0 * args.hidden, left = args.rows - r0;
        NormArgs a = args;
        a.rows = static_cast<uint32_t>(left < kRowsPerLaunch ? left : kRowsPerLaunch);
        a.x += at;
        a.out += at;
        if (a.residual) a.residual += at;
        if (a.normalized) a.normalized += at;
        if (a.residual_out) a.residual_out += at;
        switch (mode) {
            case kNormPlain: e = launch_mode<kNormPlain>(stream, a, tree); break;
            case kNormResidual: e = launch_mode<kNormResidual>(stream, a, tree); break;
            case kNormAddNorm: e = launch_mode<kNormAddNorm>(stream, a, tree); break;
            case kNormAddScale: e = launch_mode<kNormAddScale>(stream, a, tree); break;
        }
        if (e != hipSuccess) return e;
    }
    return e;
}

}  // namespace atlas
