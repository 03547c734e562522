// matvec_kernels.hip -- RMS-folded Q4_0 decode projections for gfx950.
//
// Reference semantics (bisegni/atlas, crates/atlas-metal/src/kernels.metal):
//   matvec_q4_0_16row_mv_rms           :3786-3864  one projection
//   matmul_q4_0_qkv_16row_mv_rms       :3368-3467  Q, K and V in one dispatch
//   matmul_q4_0_gate_up_16row_mv_rms   :3468-3564  gate and up in one dispatch
//   gemma4_ple_gate_gelu_f32           :803-881    the PLE input gate: plain
//       matvec, then gelu(gate) * ple[ple_offset + row] (kernels.metal:773-801)
//   callers crates/atlas-model/src/gemma4_executor.rs:2082-2119, 2502-2612
//
// One decode token: output[o] = inv_rms(x) * sum_k (x_k * w_k) * deq(W[o, k]),
// with inv_rms(x) = 1 / sqrt(sum_k x_k^2 / n + eps) -- the RMS normalisation
// of the input folded into the dispatch (its scalar applied once per output,
// as the reference does).  Without an RMS weight it is the plain Q4_0 matvec.
// Q4_0 rows are 18-byte blocks of 32 values (f16 scale d, 16 bytes; value
// j < 16 is the low nibble of byte j, value j + 16 its high nibble, minus 8).
// The reference pins these kernels with a tolerance contract against a
// normalise-then-matvec CPU oracle (crates/atlas-metal/tests/
// matvec_rms_fused_parity.rs: max-abs < 1e-3); the summation order here is
// this kernel's own, deterministic run to run.
//
// Layout on CDNA: the op streams the weight matrix once, and a vector dot of
// 4-bit codes costs more VALU work (a conversion and an FMA per weight) than
// its bytes take to arrive, so the codes meet the input on the matrix cores as
// integers (v_mfma_i32_4x4x4_16b_i8: 16 independent 4 x 4 x 4 products):
//  * each 32-value block of y = x * w becomes fixed point, rounded to steps of
//    2^-30 of the power of two above the block's largest |y| (values below about
//    2^-6 of that power lose bits to it, at most half a step each), and is split
//    into four signed byte digits; the digits of four consecutive values are one
//    word per digit, the A operand's four rows;
//  * a lane holds one weight row's block as loaded, 16 (q - 8) in the bytes of
//    eight words by a mask and a shift (q ^ 8 in a byte's high nibble is
//    16 (q - 8) in two's complement), the B operand's columns: lane l is row
//    l % 4 of the wavefront's four and block l / 4 of the pass's sixteen;
//  * eight products accumulate a block exactly in i32, one register per digit
//    and in the lane of its row; the digits meet in two halves of up to 28
//    bits, rounded as they become f32, and one fma, and the block's scale d goes
//    on with the row's running sum.
// ~45 VALU operations a block instead of ~85, 32 bytes of the input read from
// LDS per lane and block instead of 128.  Against float64, of the sum of
// |products| (root mean square over [2600, 1536]): 3.0e-9 on N(0, 1) inputs
// (vector dot 1.1e-8), 1.2e-8 with a value of 1000 in each block (3.7e-8), and
// 1.2e-8 where that value meets code 8, so that its step is all it leaves
// (vector dot, which takes the offset 8 of the whole block, 1.0e-6; the steps
// truncated instead of rounded 2.3e-8).
#include "device_common.hpp"
#include "launch.hpp"

namespace atlas {
namespace {

constexpr uint32_t kQ4Block = 18;  // bytes per 32 values
constexpr uint32_t kPassBlocks = 16, kPassRows = 4;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_block __attribute__((aligned(2)));  // a block's codes start 2 bytes into its 18

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
    return __uint_as_float(dpp_u32<CTRL>(__float_as_uint(v)));
}

// Largest value over aligned groups of 8 lanes.
__device__ __forceinline__ uint32_t group8_max(uint32_t v) {
    v = max(v, dpp_u32<0xb1>(v));         // quad_perm [1,0,3,2]
    v = max(v, dpp_u32<0x4e>(v));         // quad_perm [2,3,0,1]
    return max(v, dpp_u32<0x141>(v));     // row_half_mirror
}

// Sum over the lanes with the same lane % 4; every lane gets its total.
__device__ __forceinline__ float sum_of_row(float v) {
    v += dpp_f32<0x124>(v);  // row_ror:4
    v += dpp_f32<0x128>(v);  // row_ror:8
    v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401f));  // xor 16
    return v + __shfl_xor(v, 32, kWave);
}

// Four values as signed byte digits: word p holds digit p (weight 256^p) of
// the four, scaled by 2^shift and rounded (|v 2^shift| < 2^30).
__device__ __forceinline__ void digit_words(const f32x4 v, int shift, uint32_t (&word)[4]) {
    uint32_t t[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int q = static_cast<int>(__builtin_rintf(__builtin_ldexpf(v[i], shift)));
        // a digit d in [-128, 127] is the byte d + 128 of q + 0x808080 (the
        // top one has no bias), so clearing the bias leaves two's complement
        t[i] = (static_cast<uint32_t>(q) + 0x00808080u) ^ 0x00808080u;
    }
    // 4 x 4 byte transpose
    const uint32_t a = __builtin_amdgcn_perm(t[1], t[0], 0x05010400u), b = __builtin_amdgcn_perm(t[1], t[0], 0x07030602u);
    const uint32_t c = __builtin_amdgcn_perm(t[3], t[2], 0x05010400u), d = __builtin_amdgcn_perm(t[3], t[2], 0x07030602u);
    word[0] = __builtin_amdgcn_perm(c, a, 0x05040100u);
    word[1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
    word[2] = __builtin_amdgcn_perm(d, b, 0x05040100u);
    word[3] = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

// A block's 18 bytes behind five dwords at `p`, the 4-byte boundary at or
// below it: `high` says that it starts at the second half of the first.  The
// f16 scale comes first, the codes follow (the dwords end at most 2 bytes past
// the block: the LDS has 4 spare).
__device__ __forceinline__ void read_block(const uint32_t* p, bool high, float& d, uint32_t (&q)[4]) {
    const uint32_t w[5] = {p[0], p[1], p[2], p[3], p[4]};
    const uint32_t sel = high ? 0x07060504u : 0x05040302u;
    d = h2f(static_cast<uint16_t>(w[0] >> (high ? 16 : 0)));
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = __builtin_amdgcn_perm(w[i + 1], w[i], sel);
}

constexpr uint32_t kWaves = 4;  // wavefronts per workgroup

// LDS bytes of the input's digits and exponents, and of a wavefront's region
// for one group's rows (NBT passes of 4 x 16 blocks, 4 bytes over-read).
__host__ __device__ constexpr uint32_t plane_bytes(uint32_t nb) { return (nb * 132 + 15) & ~15u; }
__host__ __device__ constexpr uint32_t stage_bytes(int nbt) { return 4 * 16 * 18 * nbt + 16; }

// NBT passes of 16 blocks per wavefront and group of four rows.
// STAGED: a wavefront takes `groups` groups of four consecutive rows, each
// group's one contiguous span loaded with coalesced 16-byte loads and staged
// in the wavefront's LDS region while the group before it is computed.
// Otherwise (one group) the lanes load their blocks themselves: no LDS round
// trip before the dot, but 16-byte accesses 18 bytes apart, which the address
// unit takes ~225 cycles a pass over; KS wavefronts share a group's rows, NBT
// passes each.
template <int NBT, int KS, bool STAGED>
__global__ __launch_bounds__(256) void q4_0_matvec_kernel(MatvecArgs a) {
    static_assert(!STAGED || KS == 1, "a staged row belongs to one wavefront");
    constexpr int kJ = (NBT * KS * kPassBlocks * 32 / 4 + 255) / 256;  // float4 of x per thread
    constexpr int kLoads = STAGED ? (4 * 18 * NBT + 63) / 64 : NBT;  // 16-byte loads per lane and group
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ float ss_part[kWaves], bad_part[kWaves], red[KS > 1 ? kWaves * kPassRows : 1];
    const uint32_t tid = threadIdx.x, lane = tid % kWave;
    const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(tid / kWave));
    const uint32_t n = a.input_width, n4 = n / 4, nb = n / 32, row_bytes = nb * kQ4Block;
    const uint32_t groups = STAGED ? a.groups : 1u;
    const uint32_t rows = kPassRows * groups * kWaves / KS;  // rows per workgroup

    // The projection this workgroup's rows belong to (segments are tile ranges).
    const uint32_t tile = blockIdx.x;
    const uint32_t si = (a.segments > 2 && tile >= a.tile_begin[2]) ? 2 : ((a.segments > 1 && tile >= a.tile_begin[1]) ? 1 : 0);
    const uint8_t* weights = si == 0 ? a.weights[0] : (si == 1 ? a.weights[1] : a.weights[2]);
    float* out = si == 0 ? a.output[0] : (si == 1 ? a.output[1] : a.output[2]);
    const uint32_t width = si == 0 ? a.width[0] : (si == 1 ? a.width[1] : a.width[2]);
    const uint32_t begin = si == 0 ? a.tile_begin[0] : (si == 1 ? a.tile_begin[1] : a.tile_begin[2]);
    const uint32_t part = KS == 1 ? 0u : wave % KS;
    const uint32_t row0 = (tile - begin) * rows + (wave / KS) * (kPassRows * groups);  // the wavefront's first row
    const uint32_t g = lane % kPassRows, s = lane / kPassRows;
    const uint32_t b0 = KS == 1 ? 0u : min(part * (NBT * kPassBlocks), nb - 1);  // its first block of each row
    const uint32_t cnt = min(nb - b0, NBT * kPassBlocks);

    u32x4* planes = reinterpret_cast<u32x4*>(smem);                          // nb blocks x 4 digits x 8 words
    int* block_exp = reinterpret_cast<int*>(smem + nb * 128);                // nb exponents
    uint8_t* region = smem + plane_bytes(nb) + wave * stage_bytes(NBT);

    u32x4 q[kLoads];
    uint16_t qd[STAGED ? 1 : NBT];
    // rows past the end reload the last one
    auto load_group = [&](uint32_t r) {
        const uint32_t first = min(row0 + kPassRows * r, width - 1);
        if constexpr (STAGED) {
            // the last 16 bytes of a span overlap the ones before them
            const uint8_t* span = weights + static_cast<size_t>(first) * row_bytes;
            const uint32_t bytes = min(kPassRows, width - first) * row_bytes;
#pragma unroll
            for (int k = 0; k < kLoads; ++k)
                q[k] = __builtin_nontemporal_load(
                    reinterpret_cast<const u32x4_block*>(span + min(16u * (lane + 64u * k), bytes - 16u)));
        } else {
            const uint8_t* row = weights + static_cast<size_t>(min(first + g, width - 1)) * row_bytes;
#pragma unroll
            for (int t = 0; t < NBT; ++t) {
                const uint8_t* blk = row + (b0 + min(s + kPassBlocks * t, cnt - 1)) * kQ4Block;
                qd[t] = __builtin_nontemporal_load(reinterpret_cast<const uint16_t*>(blk));
                q[t] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_block*>(blk + 2));
            }
        }
    };

    // 1. input and RMS weight, then the first group's weights (the dominant
    //    stream): every load issued up front, indices clamped
    const bool rms = a.rms_weight != nullptr;
    f32x4 xv[kJ], wv[kJ];
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
        const uint32_t c = min(tid + 256u * j, n4 - 1);
        xv[j] = reinterpret_cast<const f32x4*>(a.input)[c];
        wv[j] = rms ? reinterpret_cast<const f32x4*>(a.rms_weight)[c] : f32x4{1.0f, 1.0f, 1.0f, 1.0f};
    }
    load_group(0);

    // 2. y = x * w (or x) as digits, and the sum of squares; a block is 8
    //    float4, held by 8 consecutive threads
    float ss = 0.0f;
    bool bad = false;
#pragma unroll
    for (int j = 0; j < kJ; ++j) {
        const uint32_t c = min(tid + 256u * j, n4 - 1);  // duplicates recompute the last float4
        const f32x4 x = xv[j], w = wv[j];
        f32x4 y = x;
        if (rms) y = f32x4{x.x * w.x, x.y * w.y, x.z * w.z, x.w * w.w};
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) m = max(m, __float_as_uint(y[i]) & 0x7fffffffu);
        const int e = static_cast<int>(group8_max(m) >> 23);  // |y| < 2^(e - 126) over the block
        bad = bad || e == 255;
        uint32_t word[4];
        digit_words(y, 156 - e, word);
        if (tid + 256u * j < n4) {
            if (rms) ss = ss + x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w;
            uint32_t* dst = reinterpret_cast<uint32_t*>(planes) + (c / 8) * 32 + c % 8;
#pragma unroll
            for (int p = 0; p < 4; ++p) dst[8 * p] = word[p];
            if (c % 8 == 0) block_exp[c / 8] = e - 160;  // the codes carry a factor 16
        }
    }
    ss = wave_sum_tree_f32(ss);
    const bool any_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
    if (lane == 0) {
        ss_part[wave] = ss;
        bad_part[wave] = any_bad ? __builtin_nanf("") : 0.0f;
    }
    // y and the sums are shared; the weight rows are the wavefront's own
    __syncthreads();

    // The projection is held to a tolerance, so the inverse RMS takes the
    // hardware reciprocal and reciprocal square root (each within 1 ulp):
    // rsq(sum * rcp(n) + eps), a few ulp, where the IEEE form (two divisions
    // and a square root) costs ~45 instructions per wavefront.
    float nan = bad_part[0], sum = ss_part[0];  // NaN with an infinity or NaN in y
#pragma unroll
    for (int i = 1; i < kWaves; ++i) {
        nan = nan + bad_part[i];
        sum = sum + ss_part[i];
    }
    float inv = 1.0f;
    if (rms) inv = __builtin_amdgcn_rsqf(sum * __builtin_amdgcn_rcpf(static_cast<float>(n)) + a.epsilon);

    // 3. lane (g, s): row g of each group, blocks b0 + s + 16 pass
    for (uint32_t r = 0; r < groups; ++r) {
        if constexpr (STAGED) {
            const uint32_t first = min(row0 + kPassRows * r, width - 1);
            const uint32_t bytes = min(kPassRows, width - first) * row_bytes;
#pragma unroll
            for (int k = 0; k < kLoads; ++k)
                if (16u * (lane + 64u * k) < bytes)
                    *reinterpret_cast<u32x4_block*>(region + min(16u * (lane + 64u * k), bytes - 16u)) = q[k];
            if (r + 1 < groups) load_group(r + 1);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
        // Straight-line over the passes, so their product chains overlap.  A
        // staged row's NBT passes end within 16 blocks of it: only the last
        // pass has lanes past it, which read whatever the LDS holds there
        // (inside the allocation) and are dropped; 16 blocks are 288 bytes, so
        // a lane's half-word parity is the same in every pass.  An unstaged
        // share may be shorter: its lanes repeat the last block.
        float d[NBT];
        int e[NBT];
        i32x4 p[NBT];
#pragma unroll
        for (int t = 0; t < NBT; ++t) {
            const uint32_t at = STAGED ? s + kPassBlocks * t : b0 + min(s + kPassBlocks * t, cnt - 1);
            const i32x4* src = reinterpret_cast<const i32x4*>(planes) + at * 8 + g * 2;
            const i32x4 y0 = src[0], y1 = src[1];
            e[t] = block_exp[at];
            uint32_t c[4];
            if constexpr (STAGED) {
                const uint32_t off = g * row_bytes + s * kQ4Block;
                read_block(reinterpret_cast<const uint32_t*>(region + (off & ~3u)) + t * (kPassBlocks * kQ4Block / 4),
                           (off & 2u) != 0, d[t], c);
            } else {
                d[t] = h2f(qd[t]);
#pragma unroll
                for (int w = 0; w < 4; ++w) c[w] = q[t][w];
            }
            p[t] = i32x4{0, 0, 0, 0};
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint32_t lo = ((c[w] << 4) ^ 0x80808080u) & 0xf0f0f0f0u, hi = (c[w] ^ 0x80808080u) & 0xf0f0f0f0u;
                p[t] = __builtin_amdgcn_mfma_i32_4x4x4i8(y0[w], static_cast<int>(lo), p[t], 0, 0, 0);
                p[t] = __builtin_amdgcn_mfma_i32_4x4x4i8(y1[w], static_cast<int>(hi), p[t], 0, 0, 0);
            }
        }
        float acc = 0.0f;
#pragma unroll
        for (int t = 0; t < NBT; ++t) {
            const float lo = static_cast<float>(p[t].x + (p[t].y << 8)), hi = static_cast<float>(p[t].z + (p[t].w << 8));
            const float sum = __builtin_fmaf(__builtin_ldexpf(__builtin_fmaf(hi, 65536.0f, lo), e[t]), d[t], acc);
            const bool in = (STAGED && t < NBT - 1) || part * (NBT * kPassBlocks) + s + kPassBlocks * t < nb;
            acc = in ? sum : acc;
        }
        if (STAGED) __builtin_amdgcn_wave_barrier();  // the region is read before the next group's stores
        float total = sum_of_row(acc);
        if constexpr (KS > 1) {
            if (lane < kPassRows) red[wave * kPassRows + lane] = total;
            __syncthreads();
            if (part != 0) return;
            total = 0.0f;
#pragma unroll
            for (int i = 0; i < KS; ++i) total = total + red[(wave + i) * kPassRows + g];
        }
        const uint32_t row = row0 + kPassRows * r + lane;
        if (lane < kPassRows && row < width) {
            const float v = total + nan;
            if (a.ple)  // PLE input gate: GELU of the projection times the layer's PLE slice
                out[row] = gelu_tanh_f32(v) * a.ple[a.ple_offset + row];
            else
                out[row] = rms ? v * inv : v;
        }
    }
}

template <int NBT, int KS, bool STAGED>
hipError_t launch_shape(hipStream_t stream, MatvecArgs a, uint32_t groups) {
    a.groups = static_cast<uint16_t>(groups);
    const uint32_t rows = kPassRows * groups * kWaves / KS;
    uint32_t tiles = 0;
    for (uint32_t i = 0; i < a.segments; ++i) {
        a.tile_begin[i] = tiles;
        tiles += (a.width[i] + rows - 1) / rows;
    }
    const size_t lds = plane_bytes(a.input_width / 32) + (STAGED ? kWaves * stage_bytes(NBT) : 0);
    hipLaunchKernelGGL((q4_0_matvec_kernel<NBT, KS, STAGED>), dim3(tiles), dim3(kWaves * kWave), lds, stream, a);
    return hipGetLastError();
}

// Groups of four rows per wavefront: the input's digits cost a workgroup about
// as much as one group, so the most that leave the card some 448 workgroups
// which fill their rounds over the CUs to nine tenths on average.
uint32_t staged_groups(uint32_t rows) {
    for (uint32_t groups : {4u, 2u}) {
        const uint32_t blocks = (rows + 16 * groups - 1) / (16 * groups), rounds = (blocks + 255) / 256;
        if (blocks >= 448 && 10 * blocks >= 9 * 256 * rounds) return groups;
    }
    return 1;
}

// ---------------------------------------------------------------------------
// The PLE projection of one decode token, p[o] = fl(fl(sum_k input[k] *
// W[o, k]) * scale): matvec_f16 (kernels.metal:731-740) then
// scalar_multiply_f32; the launcher follows it with the stable group norm
// (kernels.metal:897-917) in place.  Caller gemma4_executor.rs:4184-4214
// (decode: ple_projection, its scale, ple_norm).  W is F16 [rows, hidden].
// Like the reference's F16 matvec (one thread per row, its compiler's own
// contraction) the dot is held to a tolerance.
// Layout: RPW rows per wavefront, four wavefronts per workgroup; lane l
// holds input columns 8l + 512c (c < HC) in registers and streams the same
// columns of its rows with 16-byte nontemporal loads, all issued before the
// first FMA; a tree reduction per row.  (The norm as this kernel's epilogue -- the
// last workgroup of each group normalising it -- needs a device-scope
// release per workgroup, an L2 write-back on each XCD: 25 us against 8 for
// two launches.)
// ---------------------------------------------------------------------------
constexpr uint32_t kPleMaxGroups = 1024;

// Kernel parameters of the PLE projection: PleProjArgs field by field (a
// by-value struct is not preloaded into SGPRs), counts first; all 56 bytes
// arrive in user SGPRs at wave launch (kernarg preload).
#define ATLAS_PP_KPARAMS                                                                                 \
    uint32_t p_hidden, uint32_t p_width, uint32_t p_groups, float p_scale, float p_epsilon,                \
        const float* p_input, const uint16_t* p_weights, const float* p_norm_weight, float* p_output
#define ATLAS_PP_UNPACK \
    const PleProjArgs a { p_input, p_weights, p_norm_weight, p_output, p_hidden, p_width, p_groups, p_scale, p_epsilon }
#define ATLAS_PP_KARGS(a) \
    (a).hidden, (a).width, (a).groups, (a).scale, (a).epsilon, (a).input, (a).weights, (a).norm_weight, (a).output

template <int HC, int RPW>
__global__ __launch_bounds__(256) void ple_proj_f16_kernel(ATLAS_PP_KPARAMS) {
    ATLAS_PP_UNPACK;
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const uint32_t hidden = a.hidden;
    const uint32_t row0 = blockIdx.x * (4 * RPW) + wave * RPW;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

    // the rows (the dominant stream) first; a column chunk past `hidden`
    // re-reads the row's last 8 columns and meets zero inputs
    u32x4 w[RPW][HC];
#pragma unroll
    for (int i = 0; i < RPW; ++i)
#pragma unroll
        for (int c = 0; c < HC; ++c) {
            const uint32_t col = min(8 * lane + 512 * c, hidden - 8);
            w[i][c] = __builtin_nontemporal_load(
                reinterpret_cast<const u32x4*>(a.weights + static_cast<size_t>(row0 + i) * hidden + col));
        }
    float x[HC][8];
#pragma unroll
    for (int c = 0; c < HC; ++c) {
        const uint32_t col = 8 * lane + 512 * c;
        const bool in = col < hidden;
        const f32x4* src = reinterpret_cast<const f32x4*>(a.input + min(col, hidden - 8));
        const f32x4 lo = src[0], hi = src[1];
        const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
        for (int j = 0; j < 8; ++j) x[c][j] = in ? v[j] : 0.0f;
    }
    float acc[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) acc[i] = 0.0f;
#pragma unroll
    for (int c = 0; c < HC; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int i = 0; i < RPW; ++i) {
                const uint32_t word = w[i][c][j / 2];
                acc[i] = __builtin_fmaf(h2f(static_cast<uint16_t>(j & 1 ? word >> 16 : word)), x[c][j], acc[i]);
            }
    float dot[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) dot[i] = wave_sum_tree_f32(acc[i]);
    if (lane < RPW) {
        float d = dot[0];
#pragma unroll
        for (int i = 1; i < RPW; ++i) d = lane == static_cast<uint32_t>(i) ? dot[i] : d;
        a.output[row0 + lane] = d * a.scale;
    }
}

}  // namespace

uint32_t q4_0_matvec_max_input() { return 32 * 4 * 32; }

// Measured on MI355X, us (graph of launches over distinct weights): the vector
// dot that this replaces, this kernel's first form with one wavefront's four
// rows loaded by the lanes and staged, and the form kept as it is now:
//   input  rows          before  lanes  staged  now
//   1536   256 (gate)    3.12    2.97   3.04    2.50  lanes, KS = 4
//   2048   1536          2.98    3.78   3.21    2.95  lanes, KS = 2
//   4096   2048          7.14    5.43   4.67    3.93  lanes, KS = 4
//   576    3072          3.25    2.72   2.91    2.62  lanes
//   1536   2560 (QKV)    3.28    3.12   2.95    2.74  staged
//   1536   12288         5.27    4.98   4.90    4.67  staged
//   2048   16384         9.45    8.33   6.68    5.99  staged, two groups
//   3072   18432         11.8    11.8   9.58    9.25  staged
//   4096   32768         35.1    26.1   20.5    16.8  staged, four groups
// (4.5 TB/s of the weights at the last.)  A row is split between four or two
// wavefronts while that leaves each CU one workgroup (1024 and 2048 rows) and
// the row has the passes to split; from there on a second round of workgroups
// costs more than the split saves.  One projection, us: the vector dot / four
// wavefronts a row / two / one, lanes / one, staged:
//   input  rows   vector  KS=4   KS=2   lanes  staged
//   512    1024   3.02    2.99   2.98   2.83   2.90
//   512    2048   3.21    3.31   3.15   2.99   3.12
//   768    16     2.88    2.84   2.59   2.61   2.68
//   768    1024   3.06    3.04   3.14   3.08   3.30
//   768    2048   3.21    3.39   3.26   3.14   3.39
//   1024   4096   3.89    4.23   3.66   3.33   3.56
//   544    6144    -       -      -     4.04   3.75
//   1024   6144   4.43    5.02   4.10   4.00   3.97
//   32     131072  -       -      -     10.9   7.57
//   1536   1024   3.49    3.12   3.23   3.47   3.29
//   1536   2048   3.77    3.51   3.27   3.58   3.32
//   3072   1024   3.92    3.46   3.75   4.48   4.00
//   3072   1088   4.05    4.33   3.77   4.42   4.01
//   3072   2048   4.09    4.49   3.87   4.51   4.03
//   3072   2560   4.86    5.21   4.63   4.59   4.12
//   4096   1024   7.31    4.14   4.78   5.89   5.07
//   4096   2048   7.39    4.88   4.90   5.92   5.08
// More wavefronts per workgroup (8, 12 or 16 sharing the digits) were slower at
// every shape but 4096 -> 32768: the barrier waits for all of them.
hipError_t launch_q4_0_matvec(hipStream_t stream, MatvecArgs a) {
    const uint32_t nb = a.input_width / 32;
    uint64_t rows = 0;
    for (uint32_t i = 0; i < a.segments; ++i) rows += a.width[i];
    const bool few_bytes = rows <= 4096 || rows * nb <= 65536;  // the staged form pipelines more than these give it
    if (nb <= 16 && few_bytes) return launch_shape<1, 1, false>(stream, a, 1);
    if (rows <= 1024 && (nb > 32 || rows > 32))
        return nb <= 64 ? launch_shape<1, 4, false>(stream, a, 1) : launch_shape<2, 4, false>(stream, a, 1);
    if (nb <= 32 && few_bytes) return launch_shape<2, 1, false>(stream, a, 1);
    if (rows <= 2048) {
        if (nb <= 64) return launch_shape<2, 2, false>(stream, a, 1);
        return nb <= 96 ? launch_shape<3, 2, false>(stream, a, 1) : launch_shape<4, 2, false>(stream, a, 1);
    }
    const uint32_t groups = staged_groups(static_cast<uint32_t>(rows));
    switch ((nb + kPassBlocks - 1) / kPassBlocks) {
        case 1: return launch_shape<1, 1, true>(stream, a, groups);
        case 2: return launch_shape<2, 1, true>(stream, a, groups);
        case 3: return launch_shape<3, 1, true>(stream, a, groups);
        case 4: return launch_shape<4, 1, true>(stream, a, groups);
        case 5: return launch_shape<5, 1, true>(stream, a, groups);
        case 6: return launch_shape<6, 1, true>(stream, a, groups);
        case 7: return launch_shape<7, 1, true>(stream, a, groups);
        default: return launch_shape<8, 1, true>(stream, a, groups);
    }
}

uint32_t ple_projection_max_hidden() { return 512 * 8; }
uint32_t ple_projection_max_groups() { return kPleMaxGroups; }

hipError_t launch_ple_projection_f16(hipStream_t stream, const PleProjArgs& a) {
    // two rows per wavefront (eight per workgroup): 10.45 us for the op at
    // Gemma's shape, against 10.6 with one row and 11.0 with four
    constexpr int kRpw = 2;
    const dim3 grid(a.groups * a.width / (4 * kRpw));
    const uint32_t hc = (a.hidden + 511) / 512;
#define ATLAS_PLE_PROJ(H) hipLaunchKernelGGL((ple_proj_f16_kernel<H, kRpw>), grid, dim3(4 * kWave), 0, stream, \
                                            ATLAS_PP_KARGS(a))
    if (hc <= 1)
        ATLAS_PLE_PROJ(1);
    else if (hc <= 2)
        ATLAS_PLE_PROJ(2);
    else if (hc <= 3)
        ATLAS_PLE_PROJ(3);
    else if (hc <= 4)
        ATLAS_PLE_PROJ(4);
    else if (hc <= 6)
        ATLAS_PLE_PROJ(6);
    else
        ATLAS_PLE_PROJ(8);
#undef ATLAS_PLE_PROJ
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // the projection is held to a tolerance, so the norm's sum takes the tree
    return launch_rms_norm_groups_stable_f32(stream, kWide, a.output, a.norm_weight, a.width, a.groups, a.epsilon);
}

}  // namespace atlas
