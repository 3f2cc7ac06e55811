// The prefill GEMMs on the matrix cores: C[M x N] = A[M x K] . W[N x K]^T
// with the layer work that follows each product in its epilogue.
//
// A arrives as two FP16 planes written by the kernel that produced it, hi =
// fp16(a) and lo = fp16(a - hi) (a - hi is exact in FP32), W as its natural
// FP16 rows; both planes are multiplied, so products are exact and sums FP32.
//
// Operand roles: W rows are the MFMA's A operand and activation rows its B
// operand (v_mfma_f32_16x16x32_f16), so in the 16x16 result lane l holds
// activation row l % 16 and, in its 4 registers, the 4 consecutive outputs
// 4 (l / 16) .. + 3. A wave therefore has whole pieces of a row's outputs in
// its registers, and the epilogues (QK-norm, RoPE, SwiGLU, splits) run there,
// without staging C in LDS: a row sum is an in-lane sum plus exchanges with
// lanes l ^ 16 and l ^ 32.
//
// Each output element adds its K terms in one order whatever the tile: steps
// of 32 in ascending k, hi then lo in each. Results do not depend on M, on a
// row's place in a tile or on the tile shape.
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_map.hpp"
#include "half_split.hpp"
#include "kernels.hpp"
#include "prefill.hpp"

namespace qwen_hip {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// 16 bytes per lane from global memory straight into LDS at
// lds + 16 lane (lds wave-uniform); counted by vmcnt like any load.
__device__ __forceinline__ void load_lds16(const void* src, unsigned char* lds) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_global_load_lds(src, lds, 16, 0, 0);
#endif
}

// Four such loads as one opaque statement, for loops that read the LDS while
// loads into another part of it are on their way: the compiler cannot tell
// the parts apart and waits for every load it knows of before an LDS read.
// Load j fills lds + j kPitch on. base and lds (an LDS byte address)
// wave-uniform, offsets in bytes per lane. The caller waits (wait_vmcnt) before
// the data is read; the compiler's own counted waits only become stricter by the
// loads it does not see. M0 is a register that the compiler reserves, so its value
// is put back, once for the four (for each alone, prefills of 17 rows behind 3440
// took 2152 us instead of 2125).
template <int kPitch>
__device__ __forceinline__ void load4_lds16_opaque(const void* base, const unsigned* offsets, unsigned lds) {
#if defined(__HIP_DEVICE_COMPILE__)
    unsigned m0;
    asm volatile("s_mov_b32 %0, m0\n\t"
                 "s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %6\n\t"
                 "s_add_i32 m0, %1, %7\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %3, %6\n\t"
                 "s_add_i32 m0, %1, %8\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %4, %6\n\t"
                 "s_add_i32 m0, %1, %9\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, %6\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(m0)
                 : "s"(lds), "v"(offsets[0]), "v"(offsets[1]), "v"(offsets[2]), "v"(offsets[3]), "s"(base),
                   "n"(kPitch), "n"(2 * kPitch), "n"(3 * kPitch)
                 : "memory", "scc");
#endif
}
__device__ __forceinline__ unsigned lds_address(const unsigned char* p) {
#if defined(__HIP_DEVICE_COMPILE__)
    return static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const unsigned char*)p));
#else
    return 0;
#endif
}

// vmcnt <= n (expcnt and lgkmcnt unconstrained).
template <int n>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(n >= 0 && n < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
}

// lgkmcnt == 0 (this wave's LDS accesses have completed).
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4)); }

// Workgroup barrier without a memory fence: the waits before it already
// cover the direct-to-LDS loads (a fenced barrier would wait for every load
// in flight, including the later stages). The empty asm statements keep the
// compiler from moving LDS accesses across it.
__device__ __forceinline__ void stage_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// v of lane ^ 16 and of lane ^ 32, through the row swaps (register speed).
__device__ __forceinline__ int lane_xor16(int v) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return int((threadIdx.x & 16) ? r[0] : r[1]);
}
__device__ __forceinline__ int lane_xor32(int v) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return int((threadIdx.x & 32) ? r[0] : r[1]);
}
__device__ __forceinline__ float lane_xor16(float v) { return __int_as_float(lane_xor16(__float_as_int(v))); }
__device__ __forceinline__ float lane_xor32(float v) { return __int_as_float(lane_xor32(__float_as_int(v))); }
__device__ __forceinline__ double lane_xor16(double v) {
    return __hiloint2double(lane_xor16(__double2hiint(v)), lane_xor16(__double2loint(v)));
}
__device__ __forceinline__ double lane_xor32(double v) {
    return __hiloint2double(lane_xor32(__double2hiint(v)), lane_xor32(__double2loint(v)));
}

// kParts: the partial products of K range blockIdx.z, stored at C + blockIdx.z
// M N. kFold: the 4 K ranges one after the other in one workgroup, each summed
// from zero, (p0 + p1) + (p2 + p3) added into C: the sum that the row kernels
// form from kParts' ranges. Guarded: with the range guard of the down GEMM.
enum GemmKind { kStore, kParts, kPartsGuarded, kFold, kFoldGuarded, kSwiglu, kQkv };
constexpr int kKRanges = 4;

// Work fused into the epilogue. QKV (kQkv): QK-norm, RoPE and the K/V cache
// writes of engine/core.cpp:395-406. Gate/up (kSwiglu): SwiGLU, written as
// the FP16 hi / lo planes the down GEMM reads.
//
// Range guard of the FP16 split (split_exponent): A row m that its producer
// split as a * 2^-row_exp[m] has its products scaled back by 2^row_exp[m]
// (kStore, kSwiglu, kQkv). The SwiGLU
// epilogue splits each group of 8 activations with its own exponent, stored
// in act_exp [M][N / 16], and raises act_flag [M][4] (one word per K range of
// the down GEMM, cleared by the kernel before the gate/up GEMM) to the
// largest exponent in the range. The down GEMM (kParts with act_flag) runs
// its plain K loop, and a workgroup whose rows saw a nonzero flag runs the
// loop again with every group rescaled in LDS to its row's flag exponent
// and the products scaled back: a row that fits keeps its bits.
struct GemmEpilogue {
    const float* q_norm;
    const float* k_norm;
    const float* cosines;
    const float* sines;
    uint16_t* keys;
    uint16_t* values;
    int pos0;
    int context;
    uint16_t* act_hi;
    uint16_t* act_lo;
    const int* row_exp;
    int* act_flag;
    uint8_t* act_exp;
    bool add;  // kStore: C += instead of C =
};

// Tile of a workgroup: BM activation rows x BN outputs, K in stages of TK
// through a ring of NS LDS buffers. WN x WM waves run the MFMAs: wave (wn, wm)
// holds the 16-output tiles wn TN .. and the 16-row tiles wm TM ... 4 or 8 more
// waves, evenly on the SIMDs, only issue the direct global -> LDS loads: a CU accepts
// 64 bytes of loads per clock, so a stage's loads hold up the waves that issue
// them for about as long as the stage's MFMAs take, and waves that do both can
// do neither during the other.
template <int BM_, int BN_, int WN_, int WM_, int NS_, int TK_ = 64, int kLoaders_ = 4>
struct GemmTile {
    static constexpr int BM = BM_, BN = BN_, WN = WN_, WM = WM_, NS = NS_, TK = TK_;
    static constexpr int kMma = WN * WM, kLoaders = kLoaders_, kThreads = 64 * (kMma + kLoaders);
    static constexpr int TN = BN / 16 / WN, TM = BM / 16 / WM;  // 16x16 result tiles per MFMA wave
    static constexpr int SL = TK / 8;                           // 16-byte slots per operand row
    static constexpr int kSubs = TK / 32;                       // 32-column steps per stage
    static constexpr int kPlane = BM * SL, kSlots = 2 * kPlane + BN * SL;
    static constexpr int kStageBytes = 16 * kSlots;
    static constexpr int kLoads = kSlots / 64 / kLoaders;       // 1 KiB loads per loader and stage
    // Stages sent off before the first wait: 48 KiB or more, so that the first
    // one does not queue behind a whole ring.
    static constexpr int kFirst = kStageBytes >= 48 * 1024 ? 1 : (48 * 1024 + kStageBytes - 1) / kStageBytes;
    static_assert(kMma <= 8 && TN * WN * 16 == BN && TM * WM * 16 == BM, "wave grid");
    static_assert(kLoads * 64 * kLoaders == kSlots && kPlane % 64 == 0, "every loader issues the same number of loads");
    static_assert((TK == 64 || TK == 128) && NS >= 2 && NS * kStageBytes <= 160 * 1024 && (NS - 1) * kLoads < 64,
                  "stages");
};

// LDS operand rows of TK halves: piece p of row r sits in 16-byte slot
// SL r + (p ^ swz(r)), so that the 16 rows read at one piece by the lanes of
// a 16-lane group fill the 16 slots of a 256-byte bank cycle.
template <int TK>
__device__ __forceinline__ int gemm_swz(int r) {
    return TK == 64 ? ((r >> 1) ^ ((r & 1) << 2)) & 7 : r & 15;
}

// Launch arguments: the operands, the shape and the tile order.
struct GemmArgs {
    const uint16_t* Ah;
    const uint16_t* Al;
    const uint16_t* W;
    float* C;
    int M, N, K;
    int nk;  // stages of a workgroup's K range
    int mtiles, ntiles, f, per;
    unsigned magic;
};

// gate * sigmoid(gate) * up (engine/core.cpp:636-639) with e = exp(-|g|) <= 1 and
// sigmoid(g) = 1 / (1 + e), or e / (1 + e) for g < 0. One quotient step on the
// hardware reciprocal, with 1 + e carried as the two floats d + rest, rounds the
// quotient once. Measured against 64 bits (rms relative, largest in ulp): gates of
// standard deviation 0.64 3.03e-8, 2.6 ulp (0.5 + 0.5 tanh(g / 2), the reference's
// form: 3.07e-8, 4.5; 1 / (1 + exp2), divided: 4.20e-8, 3.5); |g| < 0.5 2.88e-8, 1.06
// (2.67e-8, 0.64; 4.28e-8, 2.1); -8 < g < -4, where the rounding of exp2's argument
// (1.2 x 2^-24 |g|, relative) leads, 1.8e-7, 8.0 (9.1e-6, 513; 1.8e-7, 8.8).
__device__ __forceinline__ float swiglu(float gate, float up) {
    const float e = __builtin_amdgcn_exp2f(fabsf(gate) * -1.4426950408889634f);
    const float d = 1.0f + e, rest = e - (d - 1.0f);
    const float n = gate < 0.f ? e : 1.0f, inv = __builtin_amdgcn_rcpf(d), q = n * inv;
    const float sig = __builtin_fmaf(inv, __builtin_fmaf(-rest, q, __builtin_fmaf(-d, q, n)), q);
    return gate * sig * up;
}

template <class T, int EPI>
__global__ __launch_bounds__(T::kThreads) void gemm_kernel(const GemmArgs args, const GemmEpilogue ep) {
    const uint16_t *Ah = args.Ah, *Al = args.Al, *W = args.W;
    float* C = args.C;
    const int M = args.M, N = args.N, K = args.K, nk = args.nk;
    constexpr int BM = T::BM, BN = T::BN, WN = T::WN, TN = T::TN, TM = T::TM, NS = T::NS, TK = T::TK, SL = T::SL;
    constexpr int kLoads = T::kLoads, kStageBytes = T::kStageBytes, kPlane = T::kPlane;
    constexpr bool kIsFold = EPI == kFold || EPI == kFoldGuarded;
    constexpr bool kGuarded = EPI == kPartsGuarded || EPI == kFoldGuarded;
    static_assert(EPI != kQkv || (BN == kHeadDim && TN % 2 == 0), "a QKV wave holds both channels of its RoPE pairs");
    static_assert(EPI != kSwiglu || TN % 2 == 0, "a wave of the SwiGLU epilogue holds gate and up tiles");
    // Results staged for the stores, over the ring: QKV rows (and the waves'
    // shares of the row sums), the SwiGLU planes or the C tile of the
    // workgroup; pitches of an odd number of 16-byte slots, so that 16 rows begin in
    // the 16 slots of a bank cycle.
    constexpr int kPitch = EPI == kQkv ? 4 * kHeadDim + 16 : EPI == kSwiglu ? BN + 16 : 4 * BN + 16;  // bytes
    constexpr int kOutBytes = EPI == kQkv ? BM * kPitch + 4 * BM * 8 : EPI == kSwiglu ? 2 * BM * kPitch : BM * kPitch;
    constexpr int kSmem = NS * kStageBytes > kOutBytes ? NS * kStageBytes : kOutBytes;
    static_assert(kSmem <= 160 * 1024, "LDS");
    __shared__ __align__(16) unsigned char smem[kSmem];
    const int tid = threadIdx.x, lane = tid & 63;
    const auto [mt, nt] = map_tile(blockIdx.x, args.f, args.per, args.magic);
    if (mt >= args.mtiles || nt >= args.ntiles) return;
    const int m0 = mt * BM, n0 = nt * BN;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool mma = wave < T::kMma;
    const int wn = wave % WN, wm = wave / WN % T::WM;
    const int kz = blockIdx.z * nk * TK;  // this workgroup's K range
    const int row = lane & 15, quad = lane >> 4;  // result row and output group of this lane

    // Loader i's load j fills slots 64 (i + 4 j) + lane of a stage: A hi, A lo,
    // then W rows; 64 / SL rows each. A rows past M repeat row M - 1 and are
    // never stored.
    const char* base[kLoads];  // wave-uniform
    size_t offset[kLoads];     // 64 bits: the rows of a tile may lie more than 4 GiB apart
    auto load_addresses = [&] {
        const int loader = wave - T::kMma;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int q0 = 64 * (loader + T::kLoaders * j);
            const bool is_w = q0 >= 2 * kPlane;
            const int r = (q0 - (is_w ? 2 * kPlane : q0 >= kPlane ? kPlane : 0)) / SL + lane / SL;
            const int p = (lane % SL) ^ gemm_swz<TK>(r);
            if (is_w) {
                const int r0 = r - lane / SL;
                const int first = EPI == kSwiglu ? (r0 < BN / 2 ? n0 / 2 : N / 2 + n0 / 2 - BN / 2) : n0;
                base[j] = reinterpret_cast<const char*>(W + size_t(first) * K + kz);
                offset[j] = 2 * (size_t(unsigned(r)) * unsigned(K) + unsigned(8 * p));
            } else {
                base[j] = reinterpret_cast<const char*>((q0 >= kPlane ? Al : Ah) + size_t(m0) * K + kz);
                offset[j] = 2 * (size_t(unsigned(min(r, M - 1 - m0))) * unsigned(K) + unsigned(8 * p));
            }
        }
    };
    auto issue_to = [&](int kt, int buffer) {
        unsigned char* stage = smem + buffer * kStageBytes + 1024 * (wave - T::kMma);
#pragma unroll
        for (int j = 0; j < kLoads; ++j)
            load_lds16(base[j] + offset[j] + size_t(kt) * (2 * TK), stage + 1024 * T::kLoaders * j);
    };
    auto issue = [&](int kt) { issue_to(kt, kt % NS); };
    // Waits until at most `later` whole stages of this loader's are pending.
    auto wait_stages = [&](int later) {
        if (later >= NS - 1) {
            wait_vmcnt<(NS - 1) * kLoads>();
        } else {
            switch (later) {
                case 0: wait_vmcnt<0>(); break;
                case 1: wait_vmcnt<(NS > 2 ? 1 : 0) * kLoads>(); break;
                case 2: wait_vmcnt<(NS > 3 ? 2 : 0) * kLoads>(); break;
                case 3: wait_vmcnt<(NS > 4 ? 3 : 0) * kLoads>(); break;
                case 4: wait_vmcnt<(NS > 5 ? 4 : 0) * kLoads>(); break;
                case 5: wait_vmcnt<(NS > 6 ? 5 : 0) * kLoads>(); break;
                default: wait_vmcnt<(NS > 7 ? 6 : 0) * kLoads>(); break;
            }
        }
    };

    int flagged = 0;  // nonzero: a row of the workgroup has a range flag (every wave reads them all)
    if constexpr (kGuarded) {
        for (int r = lane; r < BM; r += 64) {
            const int* flags = ep.act_flag + size_t(min(m0 + r, M - 1)) * 4;
            if constexpr (kIsFold) flagged |= flags[0] | flags[1] | flags[2] | flags[3];
            else flagged |= flags[blockIdx.z];
        }
    }
    // Stages of a K range of kFold; range 0 or 2, and the sum of ranges 0 and 1, in
    // the end of all.
    const int range = nk / kKRanges;
    floatx4 even[kIsFold ? TN : 1][kIsFold ? TM : 1], total[kIsFold ? TN : 1][kIsFold ? TM : 1];

    floatx4 acc[TN][TM];
    auto clear = [&] {
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int t = 0; t < TM; ++t) acc[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
    };
    // Operands of MFMA step `sub` of a stage: lane l reads k = 32 sub +
    // 8 (l / 16) .. + 7 of row l % 16 of each tile (tile offsets are
    // immediates: the swizzle depends on the row mod 16 only).
    auto operand_base = [&](const unsigned char* stage, int sub) {
        return stage + 16 * (SL * row + ((4 * sub + quad) ^ gemm_swz<TK>(row)));
    };
    // Output tile i of this wave starts at W row w_row(i) of the tile: gate
    // tiles then their up tiles (SwiGLU), a residue mod WN, so that tiles i and
    // i + TN / 2 are 64 rows apart (QKV), else in order.
    auto w_row = [&](int i) {
        if constexpr (EPI == kSwiglu) return 16 * (wn * (TN / 2) + i % (TN / 2)) + (i < TN / 2 ? 0 : BN / 2);
        if constexpr (EPI == kQkv) return 16 * (wn + WN * i);
        return 16 * (wn * TN + i);
    };
    auto read_w = [&](const unsigned char* at, int i) {
        return *reinterpret_cast<const half8*>(at + 32 * kPlane + 16 * SL * w_row(i));
    };
    auto read_a = [&](const unsigned char* at, int plane, int t) {
        return *reinterpret_cast<const half8*>(at + 16 * kPlane * plane + 256 * SL * (wm * TM + t));
    };
    // Half of a step: the products of one A plane, with side(c) behind MFMA c.
    auto multiply = [&](const half8 (&w)[TN], const half8 (&a)[TM], auto&& side) {
#pragma unroll
        for (int c = 0; c < TM * TN; ++c) {
            const int i = c % TN, t = c / TN;
            acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[i], a[t], acc[i][t], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            side(c);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // kFold: a range is complete; its sums, scaled by `scale(t)`, join the others.
    auto each_sum = [&](auto&& scale, auto&& join) {
        if constexpr (kIsFold) {
#pragma unroll
            for (int t = 0; t < TM; ++t) {
                const float sc = scale(t);
#pragma unroll
                for (int i = 0; i < TN; ++i) join(i, t, acc[i][t] * sc);
            }
        }
    };
    auto one = [](int) { return 1.f; };

    int rexp[TM];
    if (!mma) {
        // Loaders: stage kt is handed over by barrier kt, behind which the MFMA
        // waves have read stage kt - 1 and its buffer is refilled.
        load_addresses();
        int sent = 0;
        for (; sent < min(T::kFirst, nk); ++sent) issue(sent);
        for (int kt = 0; kt < nk; ++kt) {
            // Behind barrier kt the buffer of stage kt - 1 is free.
            if (kt == 0 && sent < nk && T::kFirst < NS) issue(sent++);
            wait_stages(sent - kt - 1);  // stage kt has landed
            stage_barrier();
#pragma unroll
            for (int more = 0; more < 2; ++more)
                if (sent < min(nk, kt + NS)) issue(sent++);
        }
    } else {
        // MFMA waves: the second half of a step reads the next step's W and A
        // hi operands, the first half its own A lo, one read behind each of
        // its first MFMAs. The barrier that hands over the next stage comes
        // between the halves of a stage's last step, when every operand of the
        // stage is in registers.
        if constexpr (EPI == kStore || EPI == kSwiglu || EPI == kQkv) {
#pragma unroll
            for (int t = 0; t < TM; ++t) rexp[t] = ep.row_exp[min(m0 + (wm * TM + t) * 16 + row, M - 1)];
        }
        clear();
        half8 w[2][TN], h[TM], l[TM];
        stage_barrier();
        {
            const unsigned char* at = operand_base(smem, 0);
#pragma unroll
            for (int i = 0; i < TN; ++i) w[0][i] = read_w(at, i);
#pragma unroll
            for (int t = 0; t < TM; ++t) h[t] = read_a(at, 0, t);
        }
        int z = 0, range_end = range;
        for (int kt = 0; kt < nk; ++kt) {
            if constexpr (kIsFold) {
                if (kt == range_end) {
                    if (z % 2 == 0) each_sum(one, [&](int i, int t, floatx4 p) { even[i][t] = p; });
                    else each_sum(one, [&](int i, int t, floatx4 p) { total[i][t] = even[i][t] + p; });
                    clear();
                    ++z;
                    range_end += range;
                }
            }
            const unsigned char* stage = smem + (kt % NS) * kStageBytes;
#pragma unroll
            for (int sub = 0; sub < T::kSubs; ++sub) {
                const unsigned char* at = operand_base(stage, sub);
                wait_lgkm0();
                __builtin_amdgcn_sched_barrier(0);
                multiply(w[sub & 1], h, [&](int c) {
                    if (c < TM) l[c] = read_a(at, 1, c);
                });
                wait_lgkm0();
                const unsigned char* next = operand_base(stage, sub + 1);
                if (sub + 1 == T::kSubs) {
                    next = operand_base(smem + ((kt + 1) % NS) * kStageBytes, 0);
                    if (kt + 1 < nk) stage_barrier();
                }
                __builtin_amdgcn_sched_barrier(0);
                // The reads behind the range's last step fetch a stage that is
                // not there: in bounds of the ring, never used.
                multiply(w[sub & 1], l, [&](int c) {
                    constexpr int kReads = TN + TM, kPer = (kReads + TM * TN - 1) / (TM * TN);
#pragma unroll
                    for (int r = c * kPer; r < (c + 1) * kPer; ++r) {
                        if (r < TM) h[r] = read_a(next, 0, r);
                        else if (r < kReads) w[(sub + 1) & 1][r - TM] = read_w(next, r - TM);
                    }
                });
            }
        }
        wait_lgkm0();
        each_sum(one, [&](int i, int t, floatx4 p) { total[i][t] = total[i][t] + (even[i][t] + p); });
    }

    // Guarded down GEMM: the loop again with each A group rescaled in LDS to its
    // row's flag exponent (exact: FP16 values times powers of two no greater
    // than 1), one stage at a time. Every wave read the same flags, so every
    // wave takes the same branch.
    bool rescaled = false;
    if constexpr (kGuarded) {
        if (__builtin_amdgcn_ballot_w64(flagged != 0) != 0) {
            rescaled = true;
            clear();
            auto row_flag = [&](int m, int z) { return ep.act_flag[size_t(min(m, M - 1)) * 4 + z]; };
            auto range_scale = [&](int z) {
                return [&, z](int t) { return pow2(row_flag(m0 + (wm * TM + t) * 16 + row, z)); };
            };
            // kFold: the sum of ranges 0 and 1 waits in LDS behind the one stage
            // (the loaders' addresses, live in this loop, leave no registers).
            static_assert(!kIsFold || kStageBytes + 4 * BM * BN <= kSmem, "parked sums");
            auto parked = [&](int i, int t) -> floatx4& {
                return *reinterpret_cast<floatx4*>(smem + kStageBytes + 16 * ((TN * t + i) * 64 * T::kMma + tid));
            };
            for (int kt = 0; kt < nk; ++kt) {
                const int z = kIsFold ? kt / range : int(blockIdx.z);
                if (kIsFold && mma && kt > 0 && kt % range == 0) {
                    each_sum(range_scale(z - 1), [&](int i, int t, floatx4 p) {
                        if (z == 2) parked(i, t) = even[i][t] + p;
                        else even[i][t] = p;
                    });
                    clear();
                }
                stage_barrier();  // every wave is done with the stage before (all loads were waited for)
                unsigned char* stage = smem;
                if (!mma) {
                    issue_to(kt, 0);
                    wait_vmcnt<0>();
                }
                stage_barrier();
                for (int q = tid; q < kPlane; q += T::kThreads) {
                    const int r = q / SL, p = (q % SL) ^ gemm_swz<TK>(r), m = min(m0 + r, M - 1);
                    const int er = row_flag(m, z);
                    if (er != 0) {
                        const int e8 = ep.act_exp[size_t(m) * (K / 8) + (kz + kt * TK) / 8 + p];
                        const float sc = pow2(e8 - er);
                        half8* hp = reinterpret_cast<half8*>(stage + 16 * q);
                        half8* lp = reinterpret_cast<half8*>(stage + 16 * (kPlane + q));
                        half8 hv = *hp, lv = *lp;
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            hv[e] = static_cast<_Float16>(static_cast<float>(hv[e]) * sc);
                            lv[e] = static_cast<_Float16>(static_cast<float>(lv[e]) * sc);
                        }
                        *hp = hv;
                        *lp = lv;
                    }
                }
                wait_lgkm0();
                stage_barrier();
                if (mma) {
#pragma unroll
                    for (int sub = 0; sub < T::kSubs; ++sub) {
                        const unsigned char* at = operand_base(stage, sub);
                        half8 w[TN], h[TM], l[TM];
#pragma unroll
                        for (int i = 0; i < TN; ++i) w[i] = read_w(at, i);
#pragma unroll
                        for (int t = 0; t < TM; ++t) {
                            h[t] = read_a(at, 0, t);
                            l[t] = read_a(at, 1, t);
                        }
                        multiply(w, h, [](int) {});
                        multiply(w, l, [](int) {});
                    }
                    wait_lgkm0();
                }
            }
            if (kIsFold && mma)
                each_sum(range_scale(kKRanges - 1),
                         [&](int i, int t, floatx4 p) { total[i][t] = parked(i, t) + (even[i][t] + p); });
        }
    }
    stage_barrier();  // every wave is done with the ring: the results are staged over it

    if constexpr (EPI <= kFoldGuarded) {
        if (mma) {
#pragma unroll
            for (int t = 0; t < TM; ++t) {
                const int r = (wm * TM + t) * 16 + row;
                float sc = 1.f;
                if constexpr (EPI == kPartsGuarded) {
                    if (rescaled) sc = pow2(ep.act_flag[size_t(min(m0 + r, M - 1)) * 4 + blockIdx.z]);
                } else if constexpr (EPI == kStore) {
                    sc = pow2(rexp[t]);
                }
#pragma unroll
                for (int i = 0; i < TN; ++i) {
                    floatx4 v;
                    if constexpr (kIsFold) v = total[i][t];
                    else v = acc[i][t];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] *= sc;
                    *reinterpret_cast<floatx4*>(smem + r * kPitch + 4 * (w_row(i) + 4 * quad)) = v;
                }
            }
        }
        __syncthreads();
#pragma unroll 4
        for (int q = tid; q < BM * (BN / 4); q += T::kThreads) {
            const int r = q / (BN / 4), c4 = q % (BN / 4), m = m0 + r;
            if (m < M) {
                floatx4 v = *reinterpret_cast<const floatx4*>(smem + r * kPitch + 16 * c4);
                floatx4* c = reinterpret_cast<floatx4*>(C + (size_t(blockIdx.z) * M + m) * N + n0) + c4;
                if constexpr (EPI == kStore || kIsFold) {
                    if (kIsFold || ep.add) {
                        const floatx4 o = *c;
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = o[e] + v[e];
                    }
                }
                *c = v;
            }
        }
    } else if constexpr (EPI == kSwiglu) {
        // Gate tiles i < TN / 2, their up tiles i + TN / 2. Lanes l and l ^ 16
        // hold a group of 8 activations: its largest magnitude sets the
        // group's exponent, and the range's flag holds the largest of those.
        if (mma) {
#pragma unroll
            for (int t = 0; t < TM; ++t) {
                const int r = (wm * TM + t) * 16 + row, m = m0 + r;
                const float sc = pow2(rexp[t]);
#pragma unroll
                for (int i = 0; i < TN / 2; ++i) {
                    float o[4], big = 0.f;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        o[e] = swiglu(acc[i][t][e] * sc, acc[i + TN / 2][t][e] * sc);
                        big = fmaxf(big, fabsf(o[e]));
                    }
                    big = fmaxf(big, lane_xor16(big));
                    const int e8 = split_exponent(big), col = w_row(i) + 4 * quad;
                    const float down = pow2(-e8);
                    half4 hi, lo;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        _Float16 h, l;
                        split_half(o[e] * down, h, l);
                        hi[e] = h;
                        lo[e] = l;
                    }
                    *reinterpret_cast<half4*>(smem + r * kPitch + 2 * col) = hi;
                    *reinterpret_cast<half4*>(smem + (BM + r) * kPitch + 2 * col) = lo;
                    if (m < M && (quad & 1) == 0) {
                        const int at = n0 / 2 + col;
                        ep.act_exp[size_t(m) * (N / 16) + at / 8] = static_cast<uint8_t>(e8);
                        if (e8 != 0) atomicMax(ep.act_flag + size_t(m) * 4 + at / (N / 8), e8);
                    }
                }
            }
        }
        __syncthreads();
#pragma unroll 4
        for (int q = tid; q < 2 * BM * (BN / 16); q += T::kThreads) {
            const int rp = q / (BN / 16), c8 = q % (BN / 16), m = m0 + rp % BM;
            if (m < M) {
                uint16_t* plane = rp < BM ? ep.act_hi : ep.act_lo;
                *reinterpret_cast<u32x4*>(plane + size_t(m) * (N / 2) + n0 / 2 + 8 * c8) =
                    *reinterpret_cast<const u32x4*>(smem + rp * kPitch + 16 * c8);
            }
        }
    } else {
        // Head nt of rows m: this lane holds channels j = w_row(i) + 4 quad + e
        // (i < TN, e < 4), so the RoPE pair (j, j + 64) is in tiles i and
        // i + TN / 2.
        const int head = nt;
        const bool is_q = head < kQHeads, is_v = head >= kQHeads + kKVHeads;
        // Row sums of the QK-norm (FP32 squares, FP64 sum, engine/core.cpp:
        // 207-215) in an order that does not depend on the tile: the tiles w
        // and w + 4 of a head together, then (0 + 1) + (2 + 3).
        constexpr int kClasses = 4 / WN;                                 // such pairs per wave
        double* sums = reinterpret_cast<double*>(smem + BM * kPitch);  // [4][BM]
        double sum[TM][kClasses];
        if (mma) {
#pragma unroll
            for (int t = 0; t < TM; ++t) {
                const float sc = pow2(rexp[t]);
#pragma unroll
                for (int i = 0; i < TN; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        acc[i][t][e] *= sc;
                        const float square = acc[i][t][e] * acc[i][t][e];
                        double& to = sum[t][i % kClasses];
                        to = i < kClasses && e == 0 ? static_cast<double>(square) : to + static_cast<double>(square);
                    }
#pragma unroll
                for (int k = 0; k < kClasses; ++k) {
                    sum[t][k] += lane_xor16(sum[t][k]);
                    sum[t][k] += lane_xor32(sum[t][k]);
                    if (WN > 1 && quad == 0) sums[(wn + WN * k) * BM + (wm * TM + t) * 16 + row] = sum[t][k];
                }
            }
        }
        if (WN > 1) __syncthreads();
        if (mma) {
#pragma unroll
            for (int t = 0; t < TM; ++t) {
                const int r = (wm * TM + t) * 16 + row, m = m0 + r;
                unsigned char* out = smem + r * kPitch;
                if (is_v) {
#pragma unroll
                    for (int i = 0; i < TN; ++i) {
                        half4 hv;
#pragma unroll
                        for (int e = 0; e < 4; ++e) hv[e] = to_half(acc[i][t][e]);
                        *reinterpret_cast<half4*>(out + 2 * (w_row(i) + 4 * quad)) = hv;
                    }
                    continue;
                }
                double c[4];
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    if constexpr (WN > 1) c[w] = sums[w * BM + r];
                    else c[w] = sum[t][w];
                }
                const float total = static_cast<float>((c[0] + c[1]) + (c[2] + c[3]));
                const float inv = 1.0f / __builtin_sqrtf(total / 128.0f + 1e-6f);
                const float* nw = (is_q ? ep.q_norm : ep.k_norm) + 4 * quad;
                const size_t rope = size_t(ep.pos0 + min(m, M - 1)) * 64 + 4 * quad;
#pragma unroll
                for (int i = 0; i < TN / 2; ++i) {
                    const floatx4 w0 = *reinterpret_cast<const floatx4*>(nw + w_row(i));
                    const floatx4 w1 = *reinterpret_cast<const floatx4*>(nw + w_row(i) + 64);
                    const floatx4 cs = *reinterpret_cast<const floatx4*>(ep.cosines + rope + w_row(i));
                    const floatx4 sn = *reinterpret_cast<const floatx4*>(ep.sines + rope + w_row(i));
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float a = (acc[i][t][e] * inv) * w0[e], b = (acc[i + TN / 2][t][e] * inv) * w1[e];
                        acc[i][t][e] = a * cs[e] - b * sn[e];
                        acc[i + TN / 2][t][e] = b * cs[e] + a * sn[e];
                    }
                }
                if constexpr (WN == 1) {
                    // Chain-permuted order (kperm): channel j = 8 s + c has its
                    // place in piece c + 8 (s / 8) at s % 8. This lane holds
                    // c = 4 (quad & 1) + e and s = 2 i + quad / 2, lane ^ 32 the
                    // other parity of s; trading the tiles i >= 4 of the lower
                    // half of the lanes for the tiles i < 4 of the upper half
                    // leaves lane half `up` with all 8 steps of the pieces
                    // c + 8 up.
                    const int piece = 4 * (quad & 1) + 8 * (lane >> 5);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float y[8];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const auto pair = __builtin_amdgcn_permlane32_swap(
                                __float_as_int(acc[i][t][e]), __float_as_int(acc[i + 4][t][e]), false, false);
                            y[2 * i] = __int_as_float(int(pair[0]));
                            y[2 * i + 1] = __int_as_float(int(pair[1]));
                        }
                        if (is_q) {
                            floatx4* q = reinterpret_cast<floatx4*>(out + 32 * (piece + e));
                            q[0] = floatx4{y[0], y[1], y[2], y[3]};
                            q[1] = floatx4{y[4], y[5], y[6], y[7]};
                        } else {
                            half8 hv;
#pragma unroll
                            for (int s = 0; s < 8; ++s) hv[s] = to_half(y[s]);
                            *reinterpret_cast<half8*>(out + 16 * (piece + e)) = hv;
                        }
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < TN; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const int at = kperm(w_row(i) + 4 * quad + e);
                            if (is_q) reinterpret_cast<float*>(out)[at] = acc[i][t][e];
                            else reinterpret_cast<uint16_t*>(out)[at] = to_half_bits(acc[i][t][e]);
                        }
                }
            }
        }
        __syncthreads();
        // Whole rows out, 16 bytes per lane.
        if (is_q) {
#pragma unroll 4
            for (int q = tid; q < BM * 32; q += T::kThreads) {
                const int r = q >> 5, c4 = q & 31;
                if (m0 + r < M)
                    reinterpret_cast<floatx4*>(C + size_t(m0 + r) * N + head * kHeadDim)[c4] =
                        *reinterpret_cast<const floatx4*>(smem + r * kPitch + 16 * c4);
            }
        } else {
            uint16_t* cache = is_v ? ep.values + size_t(head - kQHeads - kKVHeads) * ep.context * kHeadDim
                                   : ep.keys + size_t(head - kQHeads) * ep.context * kHeadDim;
#pragma unroll 4
            for (int q = tid; q < BM * 16; q += T::kThreads) {
                const int r = q >> 4, c8 = q & 15;
                if (m0 + r < M)
                    reinterpret_cast<u32x4*>(cache + size_t(ep.pos0 + m0 + r) * kHeadDim)[c8] =
                        *reinterpret_cast<const u32x4*>(smem + r * kPitch + 16 * c8);
            }
        }
    }
}

}  // namespace
}  // namespace qwen_hip
