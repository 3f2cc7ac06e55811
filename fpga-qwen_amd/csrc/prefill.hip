// Batched prefill kernels for gfx950: up to 4096 prompt rows run through
// each layer as GEMMs on the matrix cores plus row kernels
// (engine/core.cpp:353-646 with batch > 1). QK-norm, RoPE and the K/V cache
// writes run in the QKV GEMM's epilogue, SwiGLU in the gate/up GEMM's, and
// the residual adds of the K-split O and down GEMMs in the next RMSNorm.
//
// The GEMMs (prefill_gemm.hpp) multiply FP16 hi + lo planes of the FP32
// activations by natural FP16 weights: about 22 significant bits of each
// activation enter the FP32 accumulation, close to the reference's FP32 SGEMM
// (engine/core.cpp:293-294) at twice the MFMA work of a plain FP16 GEMM. Each
// output element's K order is fixed by its column, so a row's result does not
// depend on how many rows the chunk holds.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <mutex>
#include <type_traits>

#include "half_split.hpp"
#include "kernels.hpp"
#include "prefill.hpp"
#include "prefill_gemm.hpp"

namespace qwen_hip {
namespace {

__device__ __forceinline__ float h2f(uint16_t h) { return static_cast<float>(__builtin_bit_cast(_Float16, h)); }

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// x[b] = fp32(E[ids[b]]) (engine/core.cpp:382-383).
__global__ __launch_bounds__(256) void embed_rows_kernel(const int* __restrict__ ids, const uint16_t* __restrict__ E,
                                                         float* __restrict__ X) {
    const int b = blockIdx.x;
    const uint16_t* row = E + size_t(ids[b]) * kHidden;
    for (int j = threadIdx.x; j < kHidden; j += 256) X[size_t(b) * kHidden + j] = h2f(row[j]);
}

// out[b] = RMSNorm(x[b]) (engine/core.cpp:207-215): FP32 squares, FP64 sum,
// written as the FP16 hi / lo planes of the next GEMM's A operand, split as
// out * 2^-row_exp[b] (split_exponent of the row's largest magnitude; 0
// wherever the row fits FP16). With SPLITS > 0 the residual first absorbs the
// pending partial products of a K-split GEMM (parts[z][b], z < SPLITS) and is
// written back. clear_flags (optional) zeroes the row's 4 SwiGLU range flags
// ahead of the gate/up GEMM.
template <int SPLITS = 0>
__global__ __launch_bounds__(256) void rmsnorm_rows_kernel(float* __restrict__ X, const float* __restrict__ w,
                                                           uint16_t* __restrict__ out_hi,
                                                           uint16_t* __restrict__ out_lo,
                                                           const float* __restrict__ parts, int rows,
                                                           int* __restrict__ row_exp, int* __restrict__ clear_flags) {
    const int b = blockIdx.x, tid = threadIdx.x;
    // Thread t holds columns 4t .. 4t + 3 (16-byte accesses).
    float4* xr = reinterpret_cast<float4*>(X + size_t(b) * kHidden) + tid;
    float4 v4 = *xr;
    if constexpr (SPLITS > 0) {
        const size_t stride = size_t(rows) * kHidden / 4;
        const float4* pr = reinterpret_cast<const float4*>(parts + size_t(b) * kHidden) + tid;
        const float4 p0 = pr[0], p1 = pr[stride], p2 = pr[2 * stride], p3 = pr[3 * stride];
        v4.x = v4.x + ((p0.x + p1.x) + (p2.x + p3.x));
        v4.y = v4.y + ((p0.y + p1.y) + (p2.y + p3.y));
        v4.z = v4.z + ((p0.z + p1.z) + (p2.z + p3.z));
        v4.w = v4.w + ((p0.w + p1.w) + (p2.w + p3.w));
        *xr = v4;
    }
    const float v[4] = {v4.x, v4.y, v4.z, v4.w};
    double part = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float square = v[k] * v[k];
        part += static_cast<double>(square);
    }
    part = wave_sum(part);
    __shared__ double red[4];
    if ((tid & 63) == 0) red[tid >> 6] = part;
    __syncthreads();
    const float sum = static_cast<float>((red[0] + red[1]) + (red[2] + red[3]));
    const float inv = 1.0f / __builtin_sqrtf(sum / 1024.0f + 1e-6f);
    const float4 w4 = reinterpret_cast<const float4*>(w)[tid];
    const float wv[4] = {w4.x, w4.y, w4.z, w4.w};
    float n[4], big = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        n[k] = (v[k] * inv) * wv[k];
        big = fmaxf(big, fabsf(n[k]));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) big = fmaxf(big, __shfl_xor(big, off));
    __shared__ float bred[4];
    if ((tid & 63) == 0) bred[tid >> 6] = big;
    __syncthreads();
    const int e = split_exponent(fmaxf(fmaxf(bred[0], bred[1]), fmaxf(bred[2], bred[3])));
    const float down = pow2(-e);
    if (tid == 0) row_exp[b] = e;
    if (clear_flags != nullptr && tid < 4) clear_flags[size_t(b) * 4 + tid] = 0;
    uint16_t hi[4], lo[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        _Float16 h, l;
        split_half(n[k] * down, h, l);
        hi[k] = __builtin_bit_cast(uint16_t, h);
        lo[k] = __builtin_bit_cast(uint16_t, l);
    }
    const size_t at = size_t(b) * kHidden + 4 * tid;
    *reinterpret_cast<uint2*>(out_hi + at) = make_uint2(hi[0] | (unsigned(hi[1]) << 16), hi[2] | (unsigned(hi[3]) << 16));
    *reinterpret_cast<uint2*>(out_lo + at) = make_uint2(lo[0] | (unsigned(lo[1]) << 16), lo[2] | (unsigned(lo[3]) << 16));
}

// Causal attention for a prefill chunk on the matrix cores (engine/core.cpp:
// 407-605, same math as the decode path):
//   S^T = K Q^T  (A = 32 keys x 16 dims, B = Q^T as FP16 hi + lo of the FP32
//                 q, so products are exact)
//   O^T += V^T P^T (A = V^T, B = P^T as FP16 hi + lo of the FP32
//                 probabilities)
// With S^T in the 32x32 accumulator layout each lane holds 16 keys of one
// query (lane % 32), so the softmax statistics stay in the lane: one
// exchange with lane ^ 32 per tile. q and the cached keys share the
// chain-permuted channel order, which leaves q . k unchanged.
constexpr int kFaRows = 32, kFaKeys = 32, kFaccPitch = 132;
// A query keeps the reference maximum of its online softmax until a score
// exceeds it by more than this (log2 units), so probabilities stay <= 2^8 and
// most tiles need no rescaling of the output accumulators.
constexpr float kFaLazyMax = 8.f;

// Workgroup = 32 consecutive query rows x one KV head g, 8 waves (HEADS = 2):
// wave (h, s) = (wave % 2, wave / 2) runs query head 2g + h over the key tiles
// kt = s (mod 4) with its own online softmax, and the 4 key splits of each
// head are merged at the end. The two waves of a split load its K and V tiles
// together (direct global -> LDS loads, two buffers of each).
//
// A step of a wave is a matrix phase (P V of its last tile, then K Q of the
// next) and a vector phase (loads of later tiles, softmax). The two waves of a
// SIMD (splits s and s + 2) run them alternately, one barrier per phase: while
// one multiplies, the other exponentiates. With both in the same phase a step
// took 3,700 clocks (at 2,100 of MFMAs per SIMD), the vector work and the
// acceptance of 64 KiB of loads (700 clocks) serial with the MFMAs.
constexpr int kFbTileBytes = kFaKeys * kHeadDim * 2;        // one K or V tile (8 KiB)
constexpr int kFbSplitBytes = 4 * kFbTileBytes;             // a split's K buffers 0 and 1, then its V buffers
constexpr int kFbMergeBytes = 8 * kFaRows * kFaccPitch * 4; // 8 waves' outputs
constexpr int kFbLds = 4 * kFbSplitBytes > kFbMergeBytes ? 4 * kFbSplitBytes : kFbMergeBytes;
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

// K and V tiles in LDS: rows of 128 halves (sixteen 16-byte pieces), piece p
// of key row r in 16-byte slot 16 r + (p ^ fb_swz(r)). fb_swz is a bijection
// of r % 16, so 16 consecutive rows at one piece (the K operand reads) fill
// 16 distinct slots of a 256-byte bank cycle, and 4 consecutive rows (r % 4
// in bits 2-3) at 4 aligned pieces (bits 0-1) -- what 32 lanes of the V^T
// transpose load touch -- also fill 16 distinct slots.
__device__ __forceinline__ int fb_swz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }
__device__ __forceinline__ int fb_slot(int r, int p) { return 16 * r + (p ^ fb_swz(r)); }

// ds_read_b64_tr_b16 (gfx950): within each 16-lane group, lane 4a + b
// receives element b of the 8-byte chunks addressed by lanes a, a + 4,
// a + 8 and a + 12, in that order.
__device__ __forceinline__ short4_t lds_read_tr16(unsigned address) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(address));
#else
    (void)address;
    return short4_t{0, 0, 0, 0};
#endif
}
__device__ __forceinline__ half8 lds_read16(unsigned address) {
#if defined(__HIP_DEVICE_COMPILE__)
    return *(__attribute__((address_space(3))) const half8*)(address);
#else
    (void)address;
    return half8{};
#endif
}

// v - float(h[E]), exact where h[E] is v rounded: one mixed-precision FMA.
template <int E>
__device__ __forceinline__ float rest_of_half(half2 h, float v) {
#if defined(__HIP_DEVICE_COMPILE__)
    float r;
    if constexpr (E == 0)
        asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(v));
    else
        asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h), "v"(v));
    return r;
#else
    return v - static_cast<float>(h[E]);
#endif
}

// Largest value of the 8 lanes of an aligned group.
__device__ __forceinline__ float max_of_8(float v) {
    auto dpp = [](float x, auto ctrl) {
        const int b = __float_as_int(x);
        return __int_as_float(__builtin_amdgcn_update_dpp(b, b, decltype(ctrl)::value, 0xF, 0xF, false));
    };
    v = fmaxf(v, dpp(v, std::integral_constant<int, 0xB1>{}));   // quad_perm [1,0,3,2]
    v = fmaxf(v, dpp(v, std::integral_constant<int, 0x4E>{}));   // quad_perm [2,3,0,1]
    return fmaxf(v, dpp(v, std::integral_constant<int, 0x141>{}));  // the other quad of 8 lanes
}

// HEADS = 1: a workgroup of 4 waves runs one of the KV head's two query heads
// (both read its K/V tiles), for few query blocks and keys: each wave has a SIMD
// and its split's tiles to itself, so the steps need no barriers.
template <int HEADS>
__global__ __launch_bounds__(256 * HEADS) void attn_prefill_mfma_kernel(const float* __restrict__ QKV,
                                                                  const uint16_t* __restrict__ keys,
                                                                  const uint16_t* __restrict__ values,
                                                                  uint16_t* __restrict__ att_hi,
                                                                  uint16_t* __restrict__ att_lo, int rows, int pos0,
                                                                  int context, float scale) {
    __shared__ __align__(16) unsigned char lds[kFbLds];
    __shared__ float fm[4 * HEADS][kFaRows], fl[4 * HEADS][kFaRows];
    __shared__ int q_exp[HEADS][kFaRows];
    // Workgroup w runs on XCD w % 8 (round-robin dispatch): KV head g = w % 8
    // keeps every workgroup reading one head's K/V rows on one XCD, so they
    // stay in its L2; the query blocks run heaviest (latest) first.
    constexpr int kGroups = 2 / HEADS;  // workgroups of a KV head and query block
    const int nqb = gridDim.x / (kKVHeads * kGroups);
    const int g = blockIdx.x % kKVHeads, block = blockIdx.x / kKVHeads;
    const int qb = nqb - 1 - block / kGroups, first_head = 2 * g + block % kGroups;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned lds0 = __builtin_amdgcn_readfirstlane(lds_address(lds));
    const int h = wave % HEADS, sp = wave / HEADS;
    auto phase_barrier = [] { if constexpr (HEADS == 2) stage_barrier(); };
    const int col = lane & 31, hf = lane >> 5;
    const int b0 = qb * kFaRows, nrows = min(kFaRows, rows - b0);
    const int last = pos0 + b0 + nrows - 1;  // last key any query of the block attends to
    const int ntiles = last / kFaKeys + 1;
    const int nsteps = (ntiles + 3) / 4;     // steps of 4 tiles (one per split)
    const size_t head_base = size_t(g) * context;
    const int qpos = pos0 + b0 + col;        // causal limit of this lane's query
    const float scale2 = scale * 1.4426950408889634f;

    // Query rows 8 sp + lane / 8 of head h for the workgroup's Q^T operands, 16
    // channels per lane (rows past the chunk repeat its last row and are
    // never written).
    const int q_row = 8 * sp + (lane >> 3), q_lane = lane & 7;
    float qv[4][4];
    {
        const float* src = QKV + size_t(b0 + min(q_row, nrows - 1)) * kQKVRows + (first_head + h) * kHeadDim + 4 * q_lane;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 x = *reinterpret_cast<const float4*>(src + 32 * i);
            qv[i][0] = x.x, qv[i][1] = x.y, qv[i][2] = x.z, qv[i][3] = x.w;
        }
    }

    // Direct loads of step i: split sp's tile kt = 4 i + sp; load j of this
    // wave fills 16-byte slot 64 (HEADS j + h) + lane of the K or V tile; rows past
    // `last` repeat row `last` (masked). The offsets are formed ahead, for all but a
    // last tile that is not whole: the loads go out together.
    constexpr int kTileLoads = 8 / HEADS;
    unsigned ld_at[kTileLoads];  // bytes from the tile's first row
#pragma unroll
    for (int j = 0; j < kTileLoads; ++j) {
        const int q = 64 * (HEADS * j + h) + lane, r = q >> 4;
        ld_at[j] = r * (kHeadDim * 2) + 16 * ((q & 15) ^ fb_swz(r));
    }
    auto issue = [&](const uint16_t* cache, int step, int v) {
        const int kt = 4 * step + sp;
        const unsigned dst = lds0 + sp * kFbSplitBytes + (2 * v + (step & 1)) * kFbTileBytes + 1024 * h;
        const int rows_left = last - kt * kFaKeys;  // row `last` of the tile, 31 or more within
        if (rows_left < 0) return;
        const uint16_t* first = cache + (head_base + size_t(kt) * kFaKeys) * kHeadDim;
        auto load = [&](const unsigned* at) {
#pragma unroll
            for (int j = 0; j < kTileLoads; j += 4)
                load4_lds16_opaque<1024 * HEADS>(first, at + j, dst + 1024 * HEADS * j);
        };
        if (rows_left >= kFaKeys - 1) {
            load(ld_at);
        } else {
            unsigned at[kTileLoads];
#pragma unroll
            for (int j = 0; j < kTileLoads; ++j)
                at[j] = ld_at[j] - max(4 * (HEADS * j + h) + (lane >> 4) - rows_left, 0) * (kHeadDim * 2);
            load(at);
        }
    };
    issue(keys, 0, 0);

    // The queries, scaled by scale * log2(e) so that the scores come out in the
    // exp2 domain, as FP16 hi / lo planes [head][plane][row] in the V buffers
    // 1 (first used by step 1). A row whose largest magnitude reaches 65504 is
    // split as q * 2^-e (split_exponent) and its scores scaled back by 2^e.
    auto q_plane = [&](int head, int plane) { return lds + (2 * head + plane) * kFbSplitBytes + 3 * kFbTileBytes; };
    {
        float big = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                qv[i][e] = fp32_fixed(qv[i][e] * scale2);
                big = fmaxf(big, fabsf(qv[i][e]));
            }
        const int e_row = split_exponent(max_of_8(big));
        if (__builtin_amdgcn_ballot_w64(e_row != 0) != 0) {
            const float down = pow2(-e_row);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) qv[i][e] = fp32_fixed(qv[i][e] * down);
        }
        if (q_lane == 0) q_exp[h][q_row] = e_row;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            half2 hi[2], lo[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                hi[e] = __builtin_convertvector(floatx2{qv[i][2 * e], qv[i][2 * e + 1]}, half2);
                lo[e] = __builtin_convertvector(
                    floatx2{rest_of_half<0>(hi[e], qv[i][2 * e]), rest_of_half<1>(hi[e], qv[i][2 * e + 1])}, half2);
            }
            const int c = 4 * q_lane + 32 * i, at = 16 * fb_slot(q_row, c >> 3) + 2 * (c & 7);
            *reinterpret_cast<half4*>(q_plane(h, 0) + at) = half4{hi[0][0], hi[0][1], hi[1][0], hi[1][1]};
            *reinterpret_cast<half4*>(q_plane(h, 1) + at) = half4{lo[0][0], lo[0][1], lo[1][0], lo[1][1]};
        }
    }
    issue(values, 0, 1);
    issue(keys, 1, 0);
    // K tile 0 has landed: of V tile 0's and K tile 1's loads all may be pending.
    if (4 + sp < ntiles) wait_vmcnt<2 * kTileLoads>();
    else wait_vmcnt<0>();
    wait_lgkm0();
    stage_barrier();

    // Q^T operand: query b0 + col, channels 16 s + 8 hf .. + 7.
    half8 qh[8], ql[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        qh[s] = *reinterpret_cast<const half8*>(q_plane(h, 0) + 16 * fb_slot(col, 2 * s + hf));
        ql[s] = *reinterpret_cast<const half8*>(q_plane(h, 1) + 16 * fb_slot(col, 2 * s + hf));
    }
    const int eq = q_exp[h][col];
    const bool q_scaled = __builtin_amdgcn_ballot_w64(eq != 0) != 0;
    const float q_up = pow2(eq);
    float m = -INFINITY, l = 0.f;
    floatx16 acc[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;

    // Transpose-load addresses in a V tile: lane j of 16-lane group G hands
    // over key row 8 hh + 4 (G / 2) + jj / 4 (+ 16 per key step), channels
    // 32 dt + 16 (G % 2) + 4 (jj % 4) (jj = j % 16).
    const int grp = lane >> 4, jj = lane & 15;
    const int tr_row = 4 * (grp >> 1) + (jj >> 2), tr_ch = 16 * (grp & 1) + 4 * (jj & 3);
    // K operand s reads piece 2 s + hf of row col: its slot's address is k_lane
    // with 32 s folded in by xor (tile bases are multiples of 8 KiB). V operand
    // (j, dt, hh) likewise: 64 dt and 32 hh by xor, then 16 j + 8 hh rows on.
    const unsigned k_lane = lds0 + sp * kFbSplitBytes + 16 * fb_slot(col, hf);
    const unsigned v_lane = lds0 + sp * kFbSplitBytes + 2 * kFbTileBytes + 16 * fb_slot(tr_row, tr_ch >> 3) + 2 * (tr_ch & 7);
    floatx16 st;
    half8 vv[8], ph[2], pl[2];
    // P^T k slot 8 hf + i of key step j is key 16 j + 8 (i / 4) + 4 hf + i % 4;
    // transpose load hh covers keys 16 j + 8 hh + 4 hf + 0..3 of channel
    // 32 dt + lane % 32, the same order.
    auto multiply_v = [&](int j) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vv[4 * j + dt], ph[j], acc[dt], 0, 0, 0);
            acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vv[4 * j + dt], pl[j], acc[dt], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    half8 kk[8];
    auto read_k = [&](int step, int half) {
        const unsigned at = k_lane + (step & 1) * kFbTileBytes;
#pragma unroll
        for (int s = 4 * half; s < 4 * half + 4; ++s) kk[s] = lds_read16(at ^ (32 * s));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply_k = [&] {
#pragma unroll
        for (int r = 0; r < 16; ++r) st[r] = 0.f;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kk[s], qh[s], st, 0, 0, 0);
            st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kk[s], ql[s], st, 0, 0, 0);
        }
    };
    // Vector phase of step `step`: V operands into registers, then the online
    // softmax: register r of st holds key t0 + 8(r/4) + 4hf + r%4. A tile
    // entirely at or before the block's first query needs no causal mask (and
    // its maximum is finite), which saves the per-key compares and selects on
    // all but the diagonal tiles.
    auto vector_phase = [&](int step) {
        const int t0 = (4 * step + sp) * kFaKeys;
        const unsigned at = v_lane + (step & 1) * kFbTileBytes;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                const short4_t lo4 = lds_read_tr16((at ^ (64 * dt)) + 4096 * j);
                const short4_t hi4 = lds_read_tr16((at ^ (64 * dt) ^ 32) + 4096 * j + 2048);
                vv[4 * j + dt] = __builtin_bit_cast(half8, __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
            }
        __builtin_amdgcn_sched_barrier(0);
        if (q_scaled) {
#pragma unroll
            for (int r = 0; r < 16; ++r) st[r] *= q_up;
        }
        float mnew, factor, psum = 0.f;
        bool grow;
        auto softmax = [&](auto masked) {
            constexpr bool kMask = decltype(masked)::value;
            float tmax = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int t = t0 + 8 * (r >> 2) + 4 * hf + (r & 3);
                if constexpr (kMask) st[r] = t <= qpos ? st[r] : -INFINITY;
                tmax = fmaxf(tmax, st[r]);
            }
            tmax = fmaxf(tmax, lane_xor32(tmax));
            grow = tmax > m + kFaLazyMax;  // per query (both halves agree)
            mnew = grow ? tmax : m;
            factor = !grow ? 1.f : m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mnew);
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                // Both planes of two probabilities: hi rounded, lo the exact
                // rest rounded (no product feeds the conversions).
                float p[2];
#pragma unroll
                for (int e = 0; e < 2; ++e)
                    p[e] = kMask && st[r + e] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(st[r + e] - mnew);
                psum += p[0];
                psum += p[1];
                const half2 hi = __builtin_convertvector(floatx2{p[0], p[1]}, half2);
                const half2 lo = __builtin_convertvector(floatx2{rest_of_half<0>(hi, p[0]), rest_of_half<1>(hi, p[1])},
                                                         half2);
                ph[r >> 3][r & 7] = hi[0];
                ph[r >> 3][(r & 7) + 1] = hi[1];
                pl[r >> 3][r & 7] = lo[0];
                pl[r >> 3][(r & 7) + 1] = lo[1];
            }
        };
        if (t0 + kFaKeys - 1 <= pos0 + b0)
            softmax(std::false_type{});
        else
            softmax(std::true_type{});
        psum += lane_xor32(psum);
        l = l * factor + psum;
        // Rescaling by 1 changes nothing; skip it when no lane's reference moved.
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[dt][r] *= factor;
        }
        m = mnew;
    };
    // HEADS = 2: every wave passes 2 nsteps + 1 barriers: splits 2 and 3 start one
    // phase later. Only the last step can lack a tile of a split.
    const bool late = HEADS == 2 && sp >= 2;
    auto has = [&](int step) { return 4 * step + sp < ntiles; };
    wait_lgkm0();  // the Q planes are read: V tile 1 may replace them
    if (HEADS == 1 || late) stage_barrier();
    if (has(0)) {
        read_k(0, 0);
        read_k(0, 1);
        multiply_k();
    }
    if constexpr (HEADS == 1) {
        // Loads go out in two halves, V before the vector phase and K among
        // the MFMAs: all at once, 64 KiB of them per CU stalled the 4 waves
        // together.
        for (int step = 0; step + 1 < nsteps; ++step) {
            const bool next = has(step + 1);
            // V tile step has landed; K tile step + 1 may be pending.
            if (next) wait_vmcnt<kTileLoads>();
            else wait_vmcnt<0>();
            wait_lgkm0();  // V buffer step - 1 has been read
            issue(values, step + 1, 1);
            vector_phase(step);
            // K tile step + 1 has landed; V tile step + 1 may be pending.
            if (next) wait_vmcnt<kTileLoads>();
            else wait_vmcnt<0>();
            if (next) read_k(step + 1, 0);
            multiply_v(0);
            wait_lgkm0();  // K buffer step was read before
            issue(keys, step + 2, 0);
            if (next) read_k(step + 1, 1);
            multiply_v(1);
            if (next) multiply_k();
        }
    } else {
        for (int step = 0; step + 1 < nsteps; ++step) {
            wait_vmcnt<0>();  // this wave's loads of K tile step + 1 and V tile step
            wait_lgkm0();     // and its reads of K tile step (MFMAs that need them may be moved)
            phase_barrier();
            // K buffer step and V buffer step - 1 have been read by both waves.
            issue(keys, step + 2, 0);
            issue(values, step + 1, 1);
            vector_phase(step);
            wait_lgkm0();
            phase_barrier();
            if (has(step + 1)) read_k(step + 1, 0);
            multiply_v(0);
            if (has(step + 1)) read_k(step + 1, 1);
            multiply_v(1);
            if (has(step + 1)) multiply_k();
        }
    }
    wait_vmcnt<0>();
    wait_lgkm0();
    phase_barrier();
    if (has(nsteps - 1)) vector_phase(nsteps - 1);
    wait_lgkm0();
    phase_barrier();
    if (has(nsteps - 1)) {
        multiply_v(0);
        multiply_v(1);
    }
    if (HEADS == 1 || !late) stage_barrier();

    // Merge the 4 splits of each head: O^T register r of tile dt is channel
    // 32dt + 8(r/4) + 4hf + r%4 of query col.
    // Every wave is done with the K/V buffers (the barriers above).
    float(*facc)[kFaccPitch] = reinterpret_cast<float(*)[kFaccPitch]>(lds + wave * kFaRows * kFaccPitch * 4);
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; r += 4)
            *reinterpret_cast<floatx4*>(&facc[col][32 * dt + 2 * r + 4 * hf]) =
                floatx4{acc[dt][r], acc[dt][r + 1], acc[dt][r + 2], acc[dt][r + 3]};
    if (hf == 0) {
        fm[wave][col] = m;
        fl[wave][col] = l;
    }
    __syncthreads();
    // Half wave -> one query of a head at a time, 4 channels per lane.
    const int c0 = 4 * (tid & 31);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int at = (tid >> 5) + 8 * HEADS * k, hm = at / kFaRows, q = at % kFaRows;
        if (q >= nrows) continue;
        float mx = fm[hm][q];
#pragma unroll
        for (int s = 1; s < 4; ++s) mx = fmaxf(mx, fm[HEADS * s + hm][q]);
        float o[4] = {0.f, 0.f, 0.f, 0.f}, lsum = 0.f;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int w = HEADS * s + hm;
            const float e = fm[w][q] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(fm[w][q] - mx);
            lsum = __builtin_fmaf(e, fl[w][q], lsum);
            const floatx4 v = *reinterpret_cast<const floatx4*>(
                reinterpret_cast<const float*>(lds + w * kFaRows * kFaccPitch * 4) + q * kFaccPitch + c0);
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = __builtin_fmaf(e, v[i], o[i]);
        }
        half4 hi, lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // the O GEMM's A operand as FP16 hi / lo
            _Float16 hh, ll;
            split_half(o[i] / lsum, hh, ll);
            hi[i] = hh;
            lo[i] = ll;
        }
        const size_t out = size_t(b0 + q) * kQDim + (first_head + hm) * kHeadDim + c0;
        *reinterpret_cast<half4*>(att_hi + out) = hi;
        *reinterpret_cast<half4*>(att_lo + out) = lo;
    }
}

// out = x + the 4 partial products of a K-split GEMM, one row of 1024.
__global__ __launch_bounds__(256) void fold_row_kernel(const float* __restrict__ x, const float* __restrict__ parts,
                                                       float* __restrict__ out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const float* p = parts + i;
    out[i] = x[i] + ((p[0] + p[kHidden]) + (p[2 * kHidden] + p[3 * kHidden]));
}

// Tiles (by rows and outputs): MFMA wave grid (outputs x rows), LDS stages,
// stage depth, loaders. 8 loaders where the registers allow it and the tile is
// bound by its loads (1-3% over 4); the smallest tiles start faster with 4.
using Tile16x32 = GemmTile<16, 32, 1, 1, 8>;
using Tile32x32 = GemmTile<32, 32, 1, 2, 6, 128>;
using Tile32x64 = GemmTile<32, 64, 2, 2, 8>;
using Tile48x64 = GemmTile<48, 64, 2, 3, 7>;
using Tile64x64 = GemmTile<64, 64, 2, 4, 6, 64, 8>;
using Tile48x96 = GemmTile<48, 96, 3, 1, 6>;
using Tile64x96 = GemmTile<64, 96, 3, 2, 5>;
using Tile48x128 = GemmTile<48, 128, 4, 1, 5>;
using Tile64x128 = GemmTile<64, 128, 4, 2, 5, 64, 8>;
using Tile96x128 = GemmTile<96, 128, 4, 2, 4, 64, 8>;
using Tile128x128 = GemmTile<128, 128, 2, 4, 3, 64, 8>;
// Folding: the sums of the ranges take the registers of 8 loaders.
using Fold96x128 = GemmTile<96, 128, 4, 2, 4>;
using Fold128x128 = GemmTile<128, 128, 2, 4, 3>;
using Tile96x192 = GemmTile<96, 192, 3, 2, 3>;
using Tile128x192 = GemmTile<128, 192, 2, 4, 2>;
using Tile128x256 = GemmTile<128, 256, 4, 2, 2>;
using Qkv16 = GemmTile<16, 128, 4, 1, 4, 128, 8>;
using Qkv32 = GemmTile<32, 128, 4, 2, 6>;
using Qkv48 = GemmTile<48, 128, 2, 3, 5>;
using Qkv64 = GemmTile<64, 128, 2, 4, 5, 64, 8>;
using Qkv96 = GemmTile<96, 128, 1, 6, 4>;
using Qkv128 = GemmTile<128, 128, 1, 8, 3, 64, 8>;
constexpr int kTileN = 128, kTileK = 64;  // N and K granularity of the GEMM entries

template <class T, int EPI>
void launch(const uint16_t* Ah, const uint16_t* Al, const uint16_t* W, float* C, int M, int N, int K,
            hipStream_t stream, int splits, const GemmEpilogue& ep) {
    const GemmMap map(M, N, T::BM, T::BN, splits);
    const GemmArgs args{Ah, Al, W, C, M, N, K, K / splits / T::TK, map.mtiles, map.ntiles, map.f, map.per, map.magic};
    gemm_kernel<T, EPI><<<dim3(map.groups(), 1, splits), T::kThreads, 0, stream>>>(args, ep);
}

// A launch takes as many rounds as its fullest XCD has 32 workgroups, one per CU
// (of 16 x 32, two fit a CU: it is priced as if they did not); the tile with the
// least rounds x price is taken. A price is the time of a full round of that tile, in
// us: of gate/up (K 1024), of down (4 K ranges of 768; O, of 512, has the same order)
// and of QKV (K 1024); a last round that leaves CUs idle is somewhat cheaper, more so
// for the large tiles (QKV 128: 32 workgroups 14.5 us, 192 17.8 to 20, 256 21.9; gate/up
// 64 x 64: 96 9.5, 192 10.8), as fewer CUs draw on the L2s, the memory and the
// clock. Tiles of short prompts keep all CUs busy: one row tile of 128 x 128
// would leave 208 of them idle in gate/up and run 19 us. Heights of 48 and 96
// rows lie between the powers of two (whole prefill of 380 rows 2.10 -> 2.01 ms, of
// 1300 rows 4.82 -> 4.44); 96 not for the K ranges of O and down (700 rows: 96 x 128
// 13.5 / 17.3 us on all CUs, 128 x 128 on 192 of them 12.1 / 16.1, and the row kernel
// behind them 7.5 instead of 5.7).
template <int EPI>
void gemm(const uint16_t* Ah, const uint16_t* Al, const uint16_t* W, float* C, int M, int N, int K,
          hipStream_t stream, int splits = 1, const GemmEpilogue& ep = {}) {
    require(N % kTileN == 0 && K % (kTileK * splits) == 0 && M > 0 &&
                (splits == 1 || EPI == kParts || EPI == kPartsGuarded),
            "gemm: unsupported shape");
    double best = 1e30;
    void (*run)(const uint16_t*, const uint16_t*, const uint16_t*, float*, int, int, int, hipStream_t, int,
                const GemmEpilogue&) = nullptr;
    auto consider = [&]<class T>(double price) {
        if (N % T::BN != 0 || K % (T::TK * splits) != 0) return;
        const GemmMap map(M, N, T::BM, T::BN, splits);
        // A second round of small tiles of the K ranges writes its partial sums
        // behind the first's: 48 x 128 tiles at 700 rows, priced 17, cost more
        // than the 19 of one round of 128 x 128.
        if (splits > 1 && T::BM < 128 && map.rounds() > 1) return;
        const double fill = double(map.tiles(map.f) * splits - 32 * (map.rounds() - 1)) / 32;  // of the last round
        const double share = T::BM * T::BN >= 96 * 128 ? 0.28 : 0.12;
        const double cost = price * (double(map.rounds()) - share * (1 - fill * fill));
        if (cost < best) {
            best = cost;
            run = &launch<T, EPI>;
        }
    };
    if constexpr (EPI == kQkv) {  // a head per tile
        consider.template operator()<Qkv16>(7.8);
        consider.template operator()<Qkv32>(10.6);
        consider.template operator()<Qkv48>(12.6);
        consider.template operator()<Qkv64>(14.3);
        consider.template operator()<Qkv96>(20.0);
        consider.template operator()<Qkv128>(21.9);
    } else if constexpr (EPI == kParts || EPI == kPartsGuarded) {
        consider.template operator()<Tile16x32>(4.6);
        consider.template operator()<Tile32x32>(5.3);
        consider.template operator()<Tile32x64>(6.1);
        consider.template operator()<Tile48x64>(7.3);
        consider.template operator()<Tile64x64>(7.8);
        consider.template operator()<Tile48x128>(9.0);
        consider.template operator()<Tile64x128>(12.0);
        consider.template operator()<Tile128x128>(22.0);
    } else {
        consider.template operator()<Tile16x32>(6.6);
        consider.template operator()<Tile32x32>(7.7);
        consider.template operator()<Tile32x64>(8.9);
        consider.template operator()<Tile48x64>(10.3);
        consider.template operator()<Tile64x64>(10.8);
        if constexpr (EPI == kSwiglu) {
            consider.template operator()<Tile48x96>(11.9);
            consider.template operator()<Tile64x96>(13.2);
            consider.template operator()<Tile96x192>(25.8);
            consider.template operator()<Tile128x192>(29.2);
        }
        consider.template operator()<Tile64x128>(14.4);
        consider.template operator()<Tile96x128>(17.4);
        consider.template operator()<Tile128x128>(20.3);
        consider.template operator()<Tile128x256>(34.5);
    }
    run(Ah, Al, W, C, M, N, K, stream, splits, ep);
}

// O and down projections of `rows` rows into the residual x: 4 K ranges in
// their own workgroups, whose partial sums the next row kernel adds, or one
// after the other in one workgroup that adds them itself (gemm_folds). The 4
// ranges of 128 x 128 tiles fill one round up to 1024 rows; beyond, the second
// round and the partial sums (4 x rows x 4 KiB written and read) cost more than
// the longer loop: O / down with the row kernel after it at 1536 rows 25.9 / 31.8
// us in ranges, 23.1 / 29.7 folded (64 x 128 tiles, one round up to 2048 rows), at
// 3072 rows 47.3 / 60.6 and 33.1 / 46.8 (128 x 128 tiles; 96 x 128 take 27.6 where
// those take 33.6); at 1024 rows 19.4 / 23.6 and 21.5 / 27.9. Whole
// prefills of 3500 rows 12.18 -> 11.20 ms, of 3968 rows 13.47 -> 12.51.
bool gemm_folds(int rows) { return rows > kFoldRows; }

template <bool kGuarded>
void project_residual(const uint16_t* Ah, const uint16_t* Al, const uint16_t* W, float* x, float* parts, int rows, int K,
                      hipStream_t stream, const GemmEpilogue& ep) {
    constexpr int kRange = kGuarded ? kPartsGuarded : kParts, kWhole = kGuarded ? kFoldGuarded : kFold;
    if (!gemm_folds(rows))
        gemm<kRange>(Ah, Al, W, parts, rows, kHidden, K, stream, kKRanges, ep);
    else if (GemmMap(rows, kHidden, 64, 128, 1).rounds() == 1)
        launch<Tile64x128, kWhole>(Ah, Al, W, x, rows, kHidden, K, stream, 1, ep);
    else if (GemmMap(rows, kHidden, 96, 128, 1).rounds() == 1)
        launch<Fold96x128, kWhole>(Ah, Al, W, x, rows, kHidden, K, stream, 1, ep);
    else
        launch<Fold128x128, kWhole>(Ah, Al, W, x, rows, kHidden, K, stream, 1, ep);
}

// FP32 rows [M x K] -> FP16 hi / lo planes (GEMM operands handed over as
// FP32), one workgroup per row: the row is split as a * 2^-row_exp[m]
// (split_exponent of its largest magnitude). K is a multiple of 64; rows of up to
// 4096 columns stay in registers between the maximum and the split (341 x 3072: 5.4
// -> 3.6 us), longer ones are read twice.
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ A, uint16_t* __restrict__ hi,
                                                         uint16_t* __restrict__ lo, int* __restrict__ row_exp, int K) {
    typedef float piece __attribute__((ext_vector_type(4), aligned(4)));  // A is the caller's: floats, not vectors
    constexpr int kHeld = 4;  // 4-column pieces per thread
    const size_t base = size_t(blockIdx.x) * K;
    const int tid = threadIdx.x, pieces = K / 4;
    const piece* row = reinterpret_cast<const piece*>(A + base);
    floatx4 held[kHeld];
    float big = 0.f;
    auto grow = [&](floatx4 v) { big = fmaxf(fmaxf(big, fmaxf(fabsf(v[0]), fabsf(v[1]))), fmaxf(fabsf(v[2]), fabsf(v[3]))); };
#pragma unroll
    for (int k = 0; k < kHeld; ++k) held[k] = tid + 256 * k < pieces ? floatx4(row[tid + 256 * k]) : floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < kHeld; ++k) grow(held[k]);
    for (int i = tid + 256 * kHeld; i < pieces; i += 256) grow(row[i]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) big = fmaxf(big, __shfl_xor(big, off));
    __shared__ float bred[4];
    if ((tid & 63) == 0) bred[tid >> 6] = big;
    __syncthreads();
    const int e = split_exponent(fmaxf(fmaxf(bred[0], bred[1]), fmaxf(bred[2], bred[3])));
    const float down = pow2(-e);
    if (tid == 0) row_exp[blockIdx.x] = e;
    auto split = [&](floatx4 v, int i) {
        half4 h4, l4;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            _Float16 h, l;
            split_half(v[k] * down, h, l);
            h4[k] = h;
            l4[k] = l;
        }
        reinterpret_cast<half4*>(hi + base)[i] = h4;
        reinterpret_cast<half4*>(lo + base)[i] = l4;
    };
#pragma unroll
    for (int k = 0; k < kHeld; ++k)
        if (tid + 256 * k < pieces) split(held[k], tid + 256 * k);
    for (int i = tid + 256 * kHeld; i < pieces; i += 256) split(row[i], i);
}

}  // namespace

// Runs fn(hi, lo, row_exp) on FP16 hi / lo planes of the FP32 rows
// A[M x K] and their row exponents, held in device memory allocated for this
// call (an operator entry point for tests and benchmarks, not on the
// inference path), then waits for the stream.
template <class F>
static void with_planes(const float* A, int M, int K, hipStream_t stream, F&& fn) {
    require(M > 0 && K > 0, "gemm: unsupported shape");
    const size_t n = size_t(M) * K;
    auto check = [](hipError_t e, const char* what) {
        require(e == hipSuccess, std::string("HIP error: ") + hipGetErrorString(e) + " (" + what + ")");
    };
    uint16_t* planes = nullptr;
    check(hipMalloc(&planes, 2 * n * sizeof(uint16_t) + size_t(M) * sizeof(int)), "hipMalloc");
    int* row_exp = reinterpret_cast<int*>(planes + 2 * n);
    split_rows_kernel<<<M, 256, 0, stream>>>(A, planes, planes + n, row_exp, K);
    fn(planes, planes + n, row_exp);
    const hipError_t launched = hipGetLastError();
    const hipError_t done = hipStreamSynchronize(stream);
    check(hipFree(planes), "hipFree");
    check(launched, "gemm launch");
    check(done, "hipStreamSynchronize");
}

void launch_gemm(const float* A, const uint16_t* W, float* C, int M, int N, int K, bool accumulate,
                 hipStream_t stream) {
    with_planes(A, M, K, stream, [&](const uint16_t* hi, const uint16_t* lo, const int* row_exp) {
        GemmEpilogue ep{};
        ep.row_exp = row_exp;
        ep.add = accumulate;
        gemm<kStore>(hi, lo, W, C, M, N, K, stream, 1, ep);
    });
}

void launch_gemm_swiglu(const float* A, const uint16_t* W, uint16_t* act_hi, uint16_t* act_lo, uint8_t* act_exp,
                        int M, int N, int K, hipStream_t stream) {
    require(N % 256 == 0, "gemm swiglu: N must be a multiple of 256");
    int* flags = nullptr;
    require(hipMalloc(&flags, size_t(M) * 4 * sizeof(int)) == hipSuccess, "gemm swiglu: hipMalloc failed");
    const hipError_t cleared = hipMemsetAsync(flags, 0, size_t(M) * 4 * sizeof(int), stream);
    GemmEpilogue ep{};
    ep.act_hi = act_hi;
    ep.act_lo = act_lo;
    ep.act_exp = act_exp;
    ep.act_flag = flags;
    try {
        require(cleared == hipSuccess, "gemm swiglu: hipMemsetAsync failed");
        with_planes(A, M, K, stream, [&](const uint16_t* hi, const uint16_t* lo, const int* row_exp) {
            ep.row_exp = row_exp;
            gemm<kSwiglu>(hi, lo, W, nullptr, M, N, K, stream, 1, ep);
        });
    } catch (...) {
        (void)hipFree(flags);
        throw;
    }
    require(hipFree(flags) == hipSuccess, "gemm swiglu: hipFree failed");
}

// Operand planes and row exponents of launch_gemm_static: a file-scope
// device array, so the call allocates nothing. Each device holds its own copy
// at its own address (from hipGetSymbolAddress, taken once per device); host
// code uses only that address, never the array's name.
inline constexpr size_t kStaticGemmRows = kStaticGemmElements / kTileK;  // K >= 64
static __device__ __align__(256) uint16_t scratch[2 * kStaticGemmElements + 2 * kStaticGemmRows];

static uint16_t* static_planes() {
    constexpr int kMaxDevices = 64;
    static std::mutex lock;
    static uint16_t* by_device[kMaxDevices] = {};
    int device = -1;
    hipError_t e = hipGetDevice(&device);
    require(e == hipSuccess && device >= 0 && device < kMaxDevices,
            std::string("gemm static: no usable current device (") + hipGetErrorString(e) + ")");
    std::lock_guard<std::mutex> guard(lock);
    if (!by_device[device]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        require(e == hipSuccess && ptr != nullptr,
                std::string("gemm static: hipGetSymbolAddress failed (") + hipGetErrorString(e) + ")");
        by_device[device] = static_cast<uint16_t*>(ptr);
    }
    return by_device[device];
}

void launch_gemm_static(const float* A, const uint16_t* W, float* C, int M, int N, int K, bool accumulate,
                        hipStream_t stream) {
    require(M > 0 && K > 0 && N > 0 && N % kTileN == 0 && K % kTileK == 0, "gemm: unsupported shape");
    require(size_t(M) * size_t(K) <= kStaticGemmElements,
            "gemm static: M x K exceeds the 1048576 operand elements of the static planes");
    uint16_t* hi = static_planes();
    uint16_t* lo = hi + kStaticGemmElements;
    int* row_exp = reinterpret_cast<int*>(hi + 2 * kStaticGemmElements);
    split_rows_kernel<<<M, 256, 0, stream>>>(A, hi, lo, row_exp, K);
    GemmEpilogue ep{};
    ep.row_exp = row_exp;
    ep.add = accumulate;
    gemm<kStore>(hi, lo, W, C, M, N, K, stream, 1, ep);
}

void launch_attention_prefill(const float* qkv, const uint16_t* keys, const uint16_t* values, uint16_t* att_hi,
                              uint16_t* att_lo, int rows, int pos0, int context, hipStream_t stream) {
    require(rows >= 1 && rows <= kPrefillRows && pos0 >= 0 && context > 0 && pos0 + rows <= context,
            "attention: bad rows / position / context");
    const float scale = 1.0f / std::sqrt(128.0f);
    const int blocks = (rows + kFaRows - 1) / kFaRows * kKVHeads;
    // One head per workgroup while all fit one round of the 256 CUs, up to 1024
    // keys: the start and the merge halve, but a step, its vector phase no longer
    // beside another wave's MFMAs, takes longer. Whole prefills, two heads -> one:
    // 85 rows 1.357 -> 1.339 ms, 17 rows behind 612 1.359 -> 1.346, behind 1000
    // 1.463 -> 1.456, behind 1300 1.547 -> 1.564, 400 behind 3500 3.19 -> 3.28.
    if (2 * blocks <= 256 && pos0 + rows <= 1024)
        attn_prefill_mfma_kernel<1><<<2 * blocks, 256, 0, stream>>>(qkv, keys, values, att_hi, att_lo, rows, pos0,
                                                                     context, scale);
    else
        attn_prefill_mfma_kernel<2><<<blocks, 512, 0, stream>>>(qkv, keys, values, att_hi, att_lo, rows, pos0, context,
                                                                 scale);
}

void launch_prefill_chunk(const PrefillLayer* layers, const uint16_t* embed, const int* ids_dev, int rows, int pos0,
                          const float* cosines, const float* sines, int context, const PrefillScratch& s,
                          float* final_row, hipStream_t stream) {
    require(rows >= 1 && rows <= kPrefillRows, "prefill chunk: bad row count");
    embed_rows_kernel<<<rows, 256, 0, stream>>>(ids_dev, embed, s.x);
    // Where the O and down GEMMs leave their 4 K ranges apart, the row kernel
    // after each adds them to the residual, in the order in which the folding
    // GEMMs do: a row's result does not depend on the rows around it.
    auto norm = [&](const PrefillScratch& at, int count, const float* w, bool pending, int* clear_flags) {
        if (pending)
            rmsnorm_rows_kernel<kKRanges><<<count, 256, 0, stream>>>(at.x, w, at.h_hi, at.h_lo, at.part, count,
                                                                      at.row_exp, clear_flags);
        else
            rmsnorm_rows_kernel<0><<<count, 256, 0, stream>>>(at.x, w, at.h_hi, at.h_lo, nullptr, count, at.row_exp,
                                                               clear_flags);
    };
    // A layer behind its QKV GEMM, for `count` rows from position pos on (at:
    // the scratch from the first of them on).
    auto finish_layer = [&](const PrefillLayer& L, const PrefillScratch& at, int count, int pos) {
        GemmEpilogue ep{};
        ep.act_hi = at.act_hi;
        ep.act_lo = at.act_lo;
        ep.row_exp = at.row_exp;
        ep.act_flag = at.act_flag;
        ep.act_exp = at.act_exp;
        launch_attention_prefill(at.qkv, L.keys, L.values, at.att_hi, at.att_lo, count, pos, context, stream);
        // The attention output is a convex combination of FP16 values: it fits FP16 unscaled.
        project_residual<false>(at.att_hi, at.att_lo, L.o_n, at.x, at.part, count, kQDim, stream, ep);
        norm(at, count, L.post_norm, !gemm_folds(count), at.act_flag);
        gemm<kSwiglu>(at.h_hi, at.h_lo, L.gateup_n, nullptr, count, 2 * kFFN, kHidden, stream, 1, ep);
        project_residual<true>(at.act_hi, at.act_lo, L.down_n, at.x, at.part, count, kFFN, stream, ep);
    };
    // The last layer's outputs are its K/V rows and the residual of the last
    // row: behind its QKV GEMM only that row goes on (prefill of 3968 rows 11.12
    // -> 10.84 ms, of 1024 rows 3.26 -> 3.17).
    const size_t skip = size_t(rows - 1);
    const PrefillScratch last{s.x + skip * kHidden,       s.h_hi + skip * kHidden, s.h_lo + skip * kHidden,
                              s.qkv + skip * kQKVRows,    s.att_hi + skip * kQDim, s.att_lo + skip * kQDim,
                              s.act_hi + skip * kFFN,     s.act_lo + skip * kFFN,  s.part,
                              s.row_exp + skip,           s.act_flag + 4 * skip,   s.act_exp + skip * (kFFN / 8)};
    for (int l = 0; l < kLayers; ++l) {
        const PrefillLayer& L = layers[l];
        norm(s, rows, L.in_norm, l > 0 && !gemm_folds(rows), nullptr);
        GemmEpilogue ep{};
        ep.q_norm = L.q_norm;
        ep.k_norm = L.k_norm;
        ep.cosines = cosines;
        ep.sines = sines;
        ep.keys = L.keys;
        ep.values = L.values;
        ep.pos0 = pos0;
        ep.context = context;
        ep.row_exp = s.row_exp;
        gemm<kQkv>(s.h_hi, s.h_lo, L.qkv_n, s.qkv, rows, kQKVRows, kHidden, stream, 1, ep);
        if (l + 1 < kLayers) finish_layer(L, s, rows, pos0);
        else finish_layer(L, last, 1, pos0 + rows - 1);
    }
    fold_row_kernel<<<kHidden / 256, 256, 0, stream>>>(last.x, last.part, final_row);
}

}  // namespace qwen_hip
