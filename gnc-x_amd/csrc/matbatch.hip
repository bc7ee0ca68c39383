// matbatch.hip -- batched prefill product Y[B x N] = Q8(X[B x K]) . W^T.
//
// Semantics of the reference's gncx_xfold_universal_matbatch
// (csrc/gncx_llm_kernels.cpp:1495-1692): every token row of X is quantised
// on its own to per-32 int8 blocks (cpp:1506-1510), then each output is the
// same integer block dot as the matvec; the output is row-major out[t*N + m].
//
// Quantised weights (Q4_0, Q8_0, Q4_K, Q6_K) go through the fp16 matrix
// cores with exact integer operands:
//   1. act_q_kernel quantises each token row exactly as the reference does
//      and stores the quantised q as fp16 with each block's scale (and
//      launch_norm_act_q does so for the RMSNorm of a row);
//   2. matbatch_qs_stream_kernel streams the weights through registers; each
//      32-value block of a tile is one exact integer dot (Q6_K: two) on the
//      matrix cores, and the block scales are applied in fp32 on the VALU.
// Y lands within about 1e-7 relative L2 of the reference's integer block
// dots.  An int8 MFMA path would be exact too, but adds a conversion per
// output and block to that VALU work, which is what bounds the kernel.
// BF16 weights (fp32 activations, cpp:1432-1461): matbatch_bf16_kernel, the
// activations as three exact bf16 parts.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "gncx_act.h"
#include "gncx_device.h"
#include "gncx_launch.h"
#include "gncx_slots.h"

namespace gncx {
namespace {

using namespace dev;

constexpr int kThreads = 256;

// BF16 products of little work: one wave per (row, token)
__global__ __launch_bounds__(kThreads) void matbatch_rowtok_kernel(const uint8_t* __restrict w, size_t rbytes,
                                                                   const float* __restrict x, int32_t k, int32_t n,
                                                                   float* __restrict y) {
    const int lane = threadIdx.x & 63;
    const int32_t r = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
    const int32_t t = blockIdx.y;
    if (r >= n) return;
    const uint8_t* row = w + static_cast<size_t>(r) * rbytes;
    using S = Slot<kBF16>;
    const int32_t slots = S::slots(k);
    float acc = 0.0f;
    for (int32_t s = lane; s < slots; s += 64) {
        typename S::Frag f;
        typename S::Act a;
        S::load(f, PtrRow{row}, s);
        slot_act<kBF16>(a, s, nullptr, nullptr, x + static_cast<size_t>(t) * k);
        acc += S::dot(f, a, s);
    }
    acc = wave_sum(acc);
    if (lane == 0) y[static_cast<size_t>(t) * n + r] = acc;
}

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2 __attribute__((ext_vector_type(2)));

// One task's outputs (4 values of row `row`, task t of k / 4, at the
// row's 1 / s = inv): q as fp16, the block's d / s from its first lane and,
// with pq, the block's P pair.  Whole 8-lane groups call it together.
__device__ __forceinline__ void emit_q(const float4 v, int32_t t, int32_t row, int32_t k, float inv,
                                        uint2* __restrict xq, float* __restrict dxs, _Float16* __restrict pq) {
    const int32_t tasks = k / 4;
    int q0, q1, q2, q3;
    float d;
    quantize_values(v, q0, q1, q2, q3, d);
    auto h2 = [](int a, int b) {
        return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<_Float16>(a))) |
               (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<_Float16>(b))) << 16);
    };
    xq[static_cast<size_t>(row) * tasks + t] = make_uint2(h2(q0, q2), h2(q1, q3));
    if ((t & 7) == 0) dxs[static_cast<size_t>(row) * (k / 32) + (t >> 3)] = d * inv;
    if (pq) {
        // the 8 lanes of block t / 8: quad sums, then lane i adds lane 7 - i
        const int s4 = quad_sum(q0 + q1 + q2 + q3);
        const int sum = s4 + __builtin_amdgcn_mov_dpp(s4, 0x141, 0xf, 0xf, false);
        if ((t & 7) == 0) {
            const int32_t blk = t >> 3;
            const float pv = (static_cast<float>(sum) * d) * inv;
            const _Float16 ph = static_cast<_Float16>(pv);
            const _Float16 pl = static_cast<_Float16>(pv - static_cast<float>(ph));
            _Float16* pr = pq + (static_cast<size_t>(row) * (k / 256) + blk / 8) * 16 + (blk & 7);
            pr[0] = ph;
            pr[8] = pl;
        }
    }
}

// The reference's per-32 quantisation of row blockIdx.x of x (cpp:955-995):
// the quantised values q as fp16 (integers of at most 127, exact), row-major
// [B x K], and each 32-block's d / s as fp32 [B x K / 32], s the power of two
// above the row's largest |x| (stored in rscale; the product's epilogue
// multiplies it back, exactly).  Within each 8 values the order is 0 2 1 3 4
// 6 5 7, the product kernel's operand order.  With pq given (K a multiple of
// 256), also each 32-block's sum of the quantised activations, P = (sum q) *
// d / s, as an fp16 pair: per token row and 256-value super-block, 8 hi then
// 8 lo values (the Q4_K kernel's min term, cpp:1177-1178); the scale keeps P
// within fp16's range for activations of 1e5 and more (SwiGLU outputs).
// One work-group per row: the row maximum first, then 8 lanes per 32-block,
// 4 values per lane.
// With SW the row is the SwiGLU of two rows, x the gates and up the ups
// (the values gncx_swiglu_activation writes), formed as they are read.
// act_q_kernel<U> holds U float4 of x per thread in registers from the
// max pass to the quantising pass (rows up to 4 kThreads U values): the
// loads of a row are issued together, and a longer row reads its tail again.
// U = 4 covers 4096-wide rows; wider rows take U = 16, or, for the SwiGLU rows
// of the down projection up to 12288 wide, 1024 threads (NT) with U = 3, which
// keeps more of a row's loads in flight (47.9 -> 45.1 us at 2048 x 12288).
template <int U, bool SW = false, int NT = kThreads>
__global__ __launch_bounds__(NT) void act_q_kernel(const float* __restrict x, int32_t k, uint2* __restrict xq,
                                                   float* __restrict rscale, _Float16* __restrict pq,
                                                   const float* __restrict up, float* __restrict dxs) {
    __shared__ float red[NT / 64];
    const int32_t row = blockIdx.x, tasks = k / 4;
    const float4* xg = reinterpret_cast<const float4*>(x + static_cast<size_t>(row) * k);
    const float4* xu = SW ? reinterpret_cast<const float4*>(up + static_cast<size_t>(row) * k) : nullptr;
    struct Row {
        const float4* g;
        const float4* u;
        __device__ float4 operator[](int32_t t) const {
            if constexpr (!SW) {
                return g[t];
            } else {
                const float4 a = g[t], b = u[t];
                return make_float4(swiglu_value(a.x, b.x), swiglu_value(a.y, b.y), swiglu_value(a.z, b.z),
                                   swiglu_value(a.w, b.w));
            }
        }
    };
    const Row xr{xg, xu};
    auto amax4 = [](const float4 v) { return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))); };
    float4 xv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int32_t t = static_cast<int32_t>(threadIdx.x) + u * NT;
        xv[u] = t < tasks ? xr[t] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float m = 0.0f;
#pragma unroll
    for (int u = 0; u < U; ++u) m = fmaxf(m, amax4(xv[u]));
    for (int32_t t = threadIdx.x + U * NT; t < tasks; t += NT) m = fmaxf(m, amax4(xr[t]));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) m = fmaxf(m, red[w]);
    const float sc = m > 0.0f && m <= 3.0e38f ? ldexpf(1.0f, ilogbf(m) + 1) : 1.0f;  // power of two > m
    const float inv = 1.0f / sc;                                       // exact
    if (threadIdx.x == 0) rscale[row] = sc;
    auto emit = [&](const float4 v, int32_t t) { emit_q(v, t, row, k, inv, xq, dxs, pq); };
    // whole 8-lane groups take the same branches and trip counts (tasks and
    // NT are multiples of 8), as the group operations need
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int32_t t = static_cast<int32_t>(threadIdx.x) + u * NT;
        if (t < tasks) emit(xv[u], t);
    }
    for (int32_t t = threadIdx.x + U * NT; t < tasks; t += NT) emit(xr[t], t);
}

// A call's buffers in the workspace: q [B x K] and the blocks' d / s [B x K /
// 32], P (Q4_K, else null), the row scales, the split-K partials
struct QsBufs {
    _Float16* xq;
    float* dxs;
    _Float16* pq;
    float* rscale;
    float* part;
};

// up non-null: the rows are SwiGLU(x, up)
void launch_act_q(const float* x, int32_t b, int32_t k, const QsBufs& q, hipStream_t stream, const float* up) {
    uint2* o = reinterpret_cast<uint2*>(q.xq);
    if (up) {
        if (k <= 4 * 4 * kThreads)
            hipLaunchKernelGGL((act_q_kernel<4, true>), dim3(b), dim3(kThreads), 0, stream, x, k, o, q.rscale, q.pq,
                               up, q.dxs);
        else if (k <= 3 * 4 * 1024)  // up to 12288-wide rows: 16 waves, 3 float4 pairs each
            hipLaunchKernelGGL((act_q_kernel<3, true, 1024>), dim3(b), dim3(1024), 0, stream, x, k, o, q.rscale,
                               q.pq, up, q.dxs);
        else
            hipLaunchKernelGGL((act_q_kernel<16, true>), dim3(b), dim3(kThreads), 0, stream, x, k, o, q.rscale, q.pq,
                               up, q.dxs);
    } else if (b <= 512 && k > 2048 && k <= 4 * 4 * 1024) {
        // few long rows: 16 waves each (whole calls, Q6_K 14336 -> 4096 at B = 64
        // 41.7 -> 40.3 us, Q8_0 5504 -> 1438 at B = 113 30.6 -> 30.0; at B = 512
        // and for rows up to 2048 no gain)
        if (k <= 4 * 1024)
            hipLaunchKernelGGL((act_q_kernel<1, false, 1024>), dim3(b), dim3(1024), 0, stream, x, k, o, q.rscale, q.pq,
                               nullptr, q.dxs);
        else
            hipLaunchKernelGGL((act_q_kernel<4, false, 1024>), dim3(b), dim3(1024), 0, stream, x, k, o, q.rscale, q.pq,
                               nullptr, q.dxs);
    } else if (k <= 4 * 4 * kThreads) {
        hipLaunchKernelGGL((act_q_kernel<4>), dim3(b), dim3(kThreads), 0, stream, x, k, o, q.rscale, q.pq, nullptr,
                           q.dxs);
    } else {
        hipLaunchKernelGGL((act_q_kernel<16>), dim3(b), dim3(kThreads), 0, stream, x, k, o, q.rscale, q.pq, nullptr,
                           q.dxs);
    }
}

// launch_act_q of the RMSNorm of each row, after the optional residual add
// (h += r, written back), in one launch.  The norm is rmsnorm_kernel's
// (elementwise.hip) with its thread layout (1024 threads, float4 t = thread +
// 1024 j, up to 4 per thread), sum order and operation order, so the rows
// quantised are those gncx_hip_add_rmsnorm_rows / gncx_hip_rmsnorm_rows
// write; the quantisation is act_q_kernel's (a row maximum, then 8
// consecutive lanes per 32-block).
constexpr int kNaThreads = 1024;
constexpr int kNaRegs = 4;
template <bool ADD>
__global__ __launch_bounds__(kNaThreads) void norm_act_q_kernel(const float* x, const float* r, float* xo,
                                                               const float* __restrict g, int32_t k, float eps,
                                                               uint2* __restrict xq, float* __restrict dxs,
                                                               float* __restrict rscale, _Float16* __restrict pq) {
#pragma clang fp contract(off)
    __shared__ float part[kNaThreads / 64];
    __shared__ float red[kNaThreads / 64];
    const int32_t row = blockIdx.x, n4 = k / 4;
    const int tid = threadIdx.x;
    const float4* x4 = reinterpret_cast<const float4*>(x + static_cast<size_t>(row) * k);
    const float4* r4 = reinterpret_cast<const float4*>(ADD ? r + static_cast<size_t>(row) * k : nullptr);
    float4* xo4 = reinterpret_cast<float4*>(ADD ? xo + static_cast<size_t>(row) * k : nullptr);
    const float4* g4 = reinterpret_cast<const float4*>(g);
    float4 xv[kNaRegs], gv[kNaRegs];
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < kNaRegs; ++j) {
        const int32_t t = tid + kNaThreads * j;
        if (t < n4) {
            xv[j] = x4[t];
            if (ADD) {
                const float4 b = r4[t];
                xv[j] = make_float4(xv[j].x + b.x, xv[j].y + b.y, xv[j].z + b.z, xv[j].w + b.w);
                xo4[t] = xv[j];
            }
            gv[j] = g4[t];
            s += xv[j].x * xv[j].x + xv[j].y * xv[j].y + xv[j].z * xv[j].z + xv[j].w * xv[j].w;
        }
    }
    s = wave_sum(s);
    if ((tid & 63) == 0) part[tid >> 6] = s;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int w = 0; w < kNaThreads / 64; ++w) tot += part[w];
    const float inv_rms = 1.0f / sqrtf(tot / static_cast<float>(k) + eps);
    float4 yv[kNaRegs];
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < kNaRegs; ++j) {
        const int32_t t = tid + kNaThreads * j;
        yv[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (t < n4) {
            yv[j] = make_float4(xv[j].x * inv_rms * gv[j].x, xv[j].y * inv_rms * gv[j].y,
                                xv[j].z * inv_rms * gv[j].z, xv[j].w * inv_rms * gv[j].w);
            m = fmaxf(m, fmaxf(fmaxf(fabsf(yv[j].x), fabsf(yv[j].y)), fmaxf(fabsf(yv[j].z), fabsf(yv[j].w))));
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int w = 1; w < kNaThreads / 64; ++w) m = fmaxf(m, red[w]);
    const float sc = m > 0.0f && m <= 3.0e38f ? ldexpf(1.0f, ilogbf(m) + 1) : 1.0f;  // power of two > m
    const float inv = 1.0f / sc;                                                     // exact
    if (tid == 0) rscale[row] = sc;
#pragma unroll
    for (int j = 0; j < kNaRegs; ++j) {
        const int32_t t = tid + kNaThreads * j;
        if (t < n4) emit_q(yv[j], t, row, k, inv, xq, dxs, pq);
    }
}

// false when the fused form does not apply (then norm and quantise apart)
bool norm_act_fits(const float* h, const float* r, const float* gamma, int32_t k) {
    const uintptr_t al = reinterpret_cast<uintptr_t>(h) | reinterpret_cast<uintptr_t>(r) |
                         reinterpret_cast<uintptr_t>(gamma);
    return k > 0 && k % 256 == 0 && k / 4 <= kNaThreads * kNaRegs && (al & 15u) == 0;
}

void launch_norm_act_q(float* h, const float* r, const float* gamma, float eps, int32_t b, int32_t k,
                       const QsBufs& q, hipStream_t stream) {
    uint2* o = reinterpret_cast<uint2*>(q.xq);
    if (r)
        hipLaunchKernelGGL(norm_act_q_kernel<true>, dim3(b), dim3(kNaThreads), 0, stream, h, r, h, gamma, k, eps, o,
                           q.dxs, q.rscale, q.pq);
    else
        hipLaunchKernelGGL(norm_act_q_kernel<false>, dim3(b), dim3(kNaThreads), 0, stream, h, nullptr, nullptr,
                           gamma, k, eps, o, q.dxs, q.rscale, q.pq);
}

// a buffer offset past any resource (resources here are below 2^30 bytes);
// small field offsets may still be added to it without leaving int32
constexpr int32_t kMfOob = 0x7ff00000;

typedef _Float16 half4 __attribute__((ext_vector_type(4)));

// vmcnt(N) and lgkmcnt(0), then a work-group barrier with no memory fence.
// __syncthreads() says nothing of direct-to-LDS loads: in the loop the compiler
// waited there for those of later steps too (a memory round trip on every
// step), at the output of some instances for none.  Here each wave waits only
// for the loads the next step reads (vmcnt(N)) and for its own LDS writes
// (lgkmcnt(0)) before the barrier, so after it every wave sees both; the
// empty asm statements keep the compiler from moving LDS accesses across it.
template <int N>
__device__ __forceinline__ void step_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

typedef __attribute__((address_space(3))) void* lds_ptr;

// The matrices of one launch (one activation batch, the same K): x-tiles
// [tile0[i], tile0[i + 1]) are matrix i, n[i] rows, output y[i] [b x n[i]].
// A work-group picks its matrix with scalar compares and selects over the
// kernel arguments.  With split K the partials of range z are one [b x ntot]
// block, matrix i's [b x n[i]] part at b npre[i] in it (npre: rows of the
// matrices before i).
constexpr int kMaxMbMats = 4;
struct MbMats {
    const uint8_t* w[kMaxMbMats];
    float* y[kMaxMbMats];
    int32_t n[kMaxMbMats];
    int32_t tile0[kMaxMbMats];
    int32_t npre[kMaxMbMats];
    int32_t ntot;
    int32_t count;
};

// The outputs of a split-K reduce: flat partial indices [end[i - 1], end[i])
// go to y[i] (end[-1] = 0), each y[i] one contiguous [b x n] block.
struct RedMats {
    float* y[kMaxMbMats];
    size_t end[kMaxMbMats];
    int32_t count;
};

// ---- quantised weights, streamed through registers ------------------------------
//
// A work-group is 8 waves of 32 weight rows (two 16-row fragments) times 16
// TF tokens.  Each wave streams its rows' super-blocks (256 values; eight
// blocks of Q8_0 / Q4_0) straight from memory into registers, a super-block
// ahead; nothing about the weights goes through LDS but the rows' scales.
// One v_mfma_f32_16x16x32_f16 is one 32-value block of a 16 x 16 tile: lane
// l holds row (A operand, weights) or token (B, activations) l % 16 and
// values 8 kg .. 8 kg + 7 of the block, kg = kgroup(l / 16) (0 2 1 3), in the
// order 0 2 1 3 4 6 5 7 (the order in which masks pick byte pairs out of a
// dword), on both sides.
// Weights are small integers, exact in fp16, and activations the quantised q,
// so a block's product is its exact integer dot (below 2^24).  The block
// scales are applied on the VALU: S += (d_x / s) dot, where d of Q8_0 / Q4_0
// (one per row and block) goes in with d_x, and per super-block acc += d S
// (Q4_K: - dmin (m . P)).  Weights:
//   Q4_K  sc q, from the fp16 integers 1024 + q (or 1024 + 16 q for the high
//         nibbles, with sc / 16): one mask-or and one packed fma per pair
//   Q6_K  sc (q - 32) can need 12 bits (|sc| up to 128), so two products: sc
//         (l - 16) and 16 sc (u - 1) (q = l + 16 u: the 4 bits from ql, the 2
//         from qh), integers exact in fp16 for every int8 scale, from the fp16
//         values 16 + l and 4 + u with one fma each
//   Q8_0  q, Q4_0  q - 8
// Tiles of 16 x 16 rather than 32 x 32: a block is one instruction instead of
// two dependent ones, and its 4 result registers per tile leave room to scale
// one tile while the next ones multiply, and so for 128 tokens per wave, which
// halves the weights' unpacking and loads per output.
// Full calls at 4096 x 12288, B = 2048 / 512, before (32 x 32 tiles of 64
// tokens; Q8_0 and Q4_0: both operands as fp16 pairs, three products) and
// now: Q4_K 413 / 130 -> 310 / 100 us, Q6_K 665 / 213 -> 430 / 135, Q8_0 650 /
// 200 -> 412 / 140, Q4_0 635 / 196 -> 405 / 139; 64-token tiles 382 / 128 (Q4_K).
// Bound (counters, Q4_K at B = 2048): VALU issue 64% of the cycles (512 of 977
// instructions per wave and super-block, products apart, are the block scales),
// matrix cores 33%, address path 29%, LDS 26% without conflicts, at a clock of
// 2.1 GHz: no unit alone, with two waves per SIMD.  With work taken out in a
// copy (before the 16-byte loads), 335 us became 245 without the activation
// reads from LDS, 209 without products, 280 without the scales, 311 without the
// unpacking.
//
// The activations (q as fp16, d_x / s per block and, for the min term, P
// pairs) stream through three LDS stages, one super-block each, filled by
// direct-to-LDS loads two super-blocks ahead (128 tokens: two stages, which
// fill the LDS, one ahead); one barrier per super-block.
// With gridDim.z > 1 the result is a split-K partial.  It leaves through LDS,
// so that each store instruction writes one token's contiguous row range.
constexpr int kQsRows = 256;  // weight rows per work-group

typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ half2 h2_of(uint32_t v) { return __builtin_bit_cast(half2, v); }
__device__ __forceinline__ uint32_t u_of(half2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ half2 h2_all(float v) { return half2{static_cast<_Float16>(v), static_cast<_Float16>(v)}; }

// One super-block of a lane's weight row in registers.  A load costs the
// address path a cycle per lane, whatever its width (lanes of different rows
// share no line), which is what bounds the tiles of 16 and 32 tokens: so 16
// bytes a load, not the 8 that one block's operand takes of a row.  One
// work-group of 256 Q4_K rows per CU, loads alone: 2.25 -> 1.40 us per
// super-block; whole calls of 4096 x 4096 at B = 11, Q4_K 13.7 -> 12.7 us, Q8_0
// 18.6 -> 17.9, of 4096 x 14336 at B = 64, Q8_0 49.2 -> 45.0, Q4_0 46.0 -> 42.0.
// A 16-byte load holds two 8-byte pieces of a 32-byte run of the row, and four
// lane groups two runs A, B (Q4_K: two sub-block pairs): A01 A23 B01 B23.
// settle() exchanges the upper halves of lanes 0-31 with the lower halves of
// lanes 32-63: A0 A2 A1 A3 in x, y and B0 B2 B1 B3 in z, w.  So lane group g
// holds values 8 kg .. of each block, kg = kgroup(g), and reads the
// activations in that order.
// A register is loaded again, for the next super-block, as soon as its last
// block's operands are formed: load<P>(byte offset, lane group g, blocks left
// in the row) issues the loads of part P, of what block P uses last (-1: of
// what is used first).  begin(j) settles what block j is the first to use, and
// at(j, d) is dword d of its bytes.  Blocks past the row (Q8_0, Q4_0: nblk)
// read zeros.
__device__ __forceinline__ int kgroup(int g) { return (g >> 1) | ((g & 1) << 1); }
__device__ __forceinline__ void settle(u32x4& q) {
    const auto a = __builtin_amdgcn_permlane32_swap(q.x, q.z, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(q.y, q.w, false, false);
    q = u32x4{a[0], b[0], a[1], b[1]};
}
__device__ __forceinline__ uint32_t dword_of(const u32x4& q, int i) {
    return i == 0 ? q.x : i == 1 ? q.y : i == 2 ? q.z : q.w;
}
// WIDE (kQsWide): where it measured faster.  Two blocks a load hold registers
// longer: at 128 tokens Q8_0 spilled (8-18% slower) and Q4_0 (1-5%); Q6_K from
// 64 tokens is slower on rows of 2-byte alignment (2816 x 5000 at B = 2048 194
// -> 203 us, with 8-byte loads 195).
template <int TYPE, int TF>
constexpr bool kQsWide = TYPE == kQ6_K ? TF < 4 : TF < 8;
template <int TYPE, bool WIDE>
struct QsW;
template <bool WIDE>
struct QsW<kQ4_K, WIDE> {
    static constexpr int kLoads = 2;
    u32x4 q[2];  // sub-block pairs 2 i and 2 i + 1
    template <int P>
    __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& rs, int32_t off, int g, int32_t) {
        if constexpr (P >= 0 && (P & 3) == 3)
            q[P >> 2] = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16 + 64 * (P >> 2) + 16 * g, 0, 0);
    }
    __device__ __forceinline__ void begin(int j) {
        if ((j & 3) == 0) settle(q[j >> 2]);
    }
    __device__ __forceinline__ uint32_t at(int j, int d) const { return dword_of(q[j >> 2], (j & 2) + d); }
};
template <>
struct QsW<kQ6_K, true> {
    static constexpr int kLoads = 4;
    u32x4 l[2];  // ql of half i: its first and second 32 bytes
    u32x2 u[2];  // qh bytes 8 kg .. of half i (16 bytes of both would fall free with block 7 only)
    template <int P>
    __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& rs, int32_t off, int g, int32_t) {
        if constexpr (P >= 0 && (P & 3) == 3) {
            l[P >> 2] = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 64 * (P >> 2) + 16 * g, 0, 0);
            u[P >> 2] = __builtin_amdgcn_raw_buffer_load_b64(rs, off + 128 + 32 * (P >> 2) + 8 * kgroup(g), 0, 0);
        }
    }
    __device__ __forceinline__ void begin(int j) {
        if ((j & 3) == 0) settle(l[j >> 2]);
    }
    __device__ __forceinline__ uint32_t at(int j, int d) const { return dword_of(l[j >> 2], 2 * (j & 1) + d); }
    __device__ __forceinline__ uint32_t up(int j, int d) const { return d == 0 ? u[j >> 2].x : u[j >> 2].y; }
};
template <>
struct QsW<kQ6_K, false> {
    static constexpr int kLoads = 6;
    u32x2 l[4], u[2];  // ql bytes 8 kg .. of each 32, qh bytes 8 kg .. of each 32
    template <int P>
    __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& rs, int32_t off, int g, int32_t) {
        if constexpr (P >= 0 && (P & 2) == 2) {
            constexpr int i = 2 * (P >> 2) + (P & 1);
            l[i] = __builtin_amdgcn_raw_buffer_load_b64(rs, off + 8 * kgroup(g) + 32 * i, 0, 0);
            if constexpr ((P & 1) == 1)
                u[P >> 2] = __builtin_amdgcn_raw_buffer_load_b64(rs, off + 8 * kgroup(g) + 128 + 32 * (P >> 2), 0, 0);
        }
    }
    __device__ __forceinline__ void begin(int) {}
    __device__ __forceinline__ uint32_t at(int j, int d) const {
        const u32x2 v = l[2 * (j >> 2) + (j & 1)];
        return d == 0 ? v.x : v.y;
    }
    __device__ __forceinline__ uint32_t up(int j, int d) const { return d == 0 ? u[j >> 2].x : u[j >> 2].y; }
};
// Q8_0 and Q4_0 (BB bytes a block): the scales of blocks 2 g and 2 g + 1
template <int BB>
struct QsBlockScales {
    uint32_t d[2];
    __device__ __forceinline__ void load_d(const __amdgpu_buffer_rsrc_t& rs, int32_t off, int g, int32_t nblk) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
            d[e] = __builtin_amdgcn_raw_buffer_load_b16(rs, 2 * g + e < nblk ? off + BB * (2 * g + e) : kMfOob, 0, 0);
    }
};
// wide: blocks 2 i and 2 i + 1 in q[i].  Q4_0: bytes 8 (g / 2) .. of a block's
// 16, of which lane group g takes the low (g even) or high nibbles, which are
// values 8 kg .. again
template <int BB>
struct QsWideBlocks : QsBlockScales<BB> {
    static constexpr int kLoads = 6;
    u32x4 q[4];
    template <int P>
    __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& rs, int32_t off, int g, int32_t nblk) {
        if constexpr (P == -1) this->load_d(rs, off, g, nblk);
        else if constexpr ((P & 1) == 1) {
            const int blk = P - 1 + (g >> 1), at = BB == 34 ? 16 * (g & 1) : 0;
            q[P >> 1] = __builtin_amdgcn_raw_buffer_load_b128(rs, blk < nblk ? off + BB * blk + 2 + at : kMfOob, 0, 0);
        }
    }
    __device__ __forceinline__ void begin(int j) {
        if ((j & 1) == 0) settle(q[j >> 1]);
    }
    __device__ __forceinline__ uint32_t at(int j, int d) const { return dword_of(q[j >> 1], 2 * (j & 1) + d); }
};
// one block's 8 bytes a load
template <int BB>
struct QsNarrowBlocks : QsBlockScales<BB> {
    static constexpr int kLoads = 10;
    u32x2 q[8];
    template <int P>
    __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& rs, int32_t off, int g, int32_t nblk) {
        if constexpr (P == -1) this->load_d(rs, off, g, nblk);
        else {
            const int at = BB == 34 ? 8 * kgroup(g) : 8 * (g >> 1);
            q[P] = __builtin_amdgcn_raw_buffer_load_b64(rs, P < nblk ? off + BB * P + 2 + at : kMfOob, 0, 0);
        }
    }
    __device__ __forceinline__ void begin(int) {}
    __device__ __forceinline__ uint32_t at(int j, int d) const { return d == 0 ? q[j].x : q[j].y; }
};
template <>
struct QsW<kQ8_0, true> : QsWideBlocks<34> {};
template <>
struct QsW<kQ8_0, false> : QsNarrowBlocks<34> {};
template <>
struct QsW<kQ4_0, true> : QsWideBlocks<18> {};
template <>
struct QsW<kQ4_0, false> : QsNarrowBlocks<18> {};

// The super-block scales of both fragments' rows, one load for the wave (as
// above): lane l reads row l % 32, row l % 16 of fragment l / 16 % 2, and
// spread() gives every lane the scales of its row of each fragment, odd lane
// groups of one copy exchanged with even ones of another.
template <int TYPE>
struct QsH {  // Q8_0, Q4_0: the block scales are in QsW
    static constexpr int kLoads = 0;
    __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t&, int32_t) {}
};
template <>
struct QsH<kQ4_K> {
    static constexpr int kLoads = 1;
    u32x4 h;  // d and dmin, the 12 scale bytes
    __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& rs, int32_t off) {
        h = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
    }
};
template <>
struct QsH<kQ6_K> {
    static constexpr int kLoads = 2;
    u32x4 h;  // the 16 scales
    uint32_t d;
    __device__ __forceinline__ void load(const __amdgpu_buffer_rsrc_t& rs, int32_t off) {
        h = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 192, 0, 0);
        d = __builtin_amdgcn_raw_buffer_load_b16(rs, off + 208, 0, 0);
    }
};
__device__ __forceinline__ void spread(const u32x4& h, u32x4 (&o)[2]) {
    const auto x = __builtin_amdgcn_permlane16_swap(h.x, h.x, false, false);
    const auto y = __builtin_amdgcn_permlane16_swap(h.y, h.y, false, false);
    const auto z = __builtin_amdgcn_permlane16_swap(h.z, h.z, false, false);
    const auto w = __builtin_amdgcn_permlane16_swap(h.w, h.w, false, false);
    o[0] = u32x4{x[0], y[0], z[0], w[0]};
    o[1] = u32x4{x[1], y[1], z[1], w[1]};
}

// (v & mask) | e as one v_and_or_b32: with e hidden in a vector register and
// the mask in a scalar one (two literals would take two instructions)
__device__ __forceinline__ uint32_t in_vgpr(uint32_t v) {
    asm("" : "+v"(v));
    return v;
}

// The A operands of a lane's row for one super-block: prepare(h, g) unpacks
// what all blocks share from the row's scales, get(w, g, j, d, o) forms dword d
// (0, 1; 0 first) of block j's operand, 4 of its 8 values (o.b: Q6_K's second
// product).
struct QsOut {
    uint32_t a[4], b[4];
};
template <int TYPE>
struct QsOperand;
template <>
struct QsOperand<kQ4_K> {
    uint32_t sc[2], mn[2];  // 6-bit scales and mins of sub-blocks 0-3 and 4-7, a byte each
    uint32_t e;
    half2 s, m;  // of the block being formed
    __device__ __forceinline__ void prepare(const u32x4& h, int) {
        e = in_vgpr(0x64006400u);
        sc[0] = h.y & 0x3f3f3f3fu;
        mn[0] = h.z & 0x3f3f3f3fu;
        sc[1] = (h.w & 0x0f0f0f0fu) | ((h.y >> 2) & 0x30303030u);
        mn[1] = ((h.w >> 4) & 0x0f0f0f0fu) | ((h.z >> 2) & 0x30303030u);
    }
    template <class W>
    __device__ __forceinline__ void get(W& w, int, int j, int d, QsOut& o) {
        if (d == 0) {
            w.begin(j);
            const uint32_t sel = 0x04000400u | (0x00010001u * static_cast<uint32_t>(j & 3));
            const half2 t = h2_of(__builtin_amdgcn_perm(0x64646464u, sc[j >> 2], sel));  // 1024 + sc
            // low nibbles sit under the exponent of 1024 as they are, high ones times 16
            s = (j & 1) == 0 ? t + h2_all(-1024.0f) : __builtin_elementwise_fma(t, h2_all(0.0625f), h2_all(-64.0f));
            m = s * h2_all(-1024.0f);
        }
        const uint32_t mask = (j & 1) == 0 ? 0x000f000fu : 0x00f000f0u;
        const uint32_t v = w.at(j, d);
        o.a[2 * d] = u_of(__builtin_elementwise_fma(h2_of((v & mask) | e), s, m));
        o.a[2 * d + 1] = u_of(__builtin_elementwise_fma(h2_of(((v >> 8) & mask) | e), s, m));
    }
};
template <>
struct QsOperand<kQ6_K> {
    uint32_t sc[4];  // scale + 128 of blocks 2 i and 2 i + 1 in bytes 0 and 2
    uint32_t e1, e2;
    half2 s1, m1, s2, m2;
    __device__ __forceinline__ void prepare(const u32x4& h, int g) {
        e1 = in_vgpr(0x4c004c00u);
        e2 = in_vgpr(0x44004400u);
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[i] = (dword_of(h, i) ^ 0x80808080u) >> (8 * (kgroup(g) >> 1));
    }
    template <class W>
    __device__ __forceinline__ void get(W& w, int, int j, int d, QsOut& o) {
        const int gr = j & 3;
        if (d == 0) {
            w.begin(j);
            const uint32_t sel = (j & 1) == 0 ? 0x04000400u : 0x04020402u;
            s1 = h2_of(__builtin_amdgcn_perm(0x64646464u, sc[j >> 1], sel)) + h2_all(-1152.0f);
            m1 = s1 * h2_all(-32.0f);
            s2 = s1 * h2_all(16.0f);
            m2 = s1 * h2_all(-80.0f);
        }
        const uint32_t l = w.at(j, d), u = w.up(j, d);
        // the nibbles of bytes 0, 2 / 1, 3 at bits 6..9 of each half: 16 + l
        const uint32_t l0 = gr < 2 ? l << 6 : l << 2, l1 = gr < 2 ? l >> 2 : l >> 6;
        o.a[2 * d] = u_of(__builtin_elementwise_fma(h2_of((l0 & 0x03c003c0u) | e1), s1, m1));
        o.a[2 * d + 1] = u_of(__builtin_elementwise_fma(h2_of((l1 & 0x03c003c0u) | e1), s1, m1));
        // the 2-bit values at bits 8, 9: 4 + u
        const uint32_t u0 = u << (8 - 2 * gr), u1 = u >> (2 * gr);
        o.b[2 * d] = u_of(__builtin_elementwise_fma(h2_of((u0 & 0x03000300u) | e2), s2, m2));
        o.b[2 * d + 1] = u_of(__builtin_elementwise_fma(h2_of((u1 & 0x03000300u) | e2), s2, m2));
    }
};
template <>
struct QsOperand<kQ8_0> {
    __device__ __forceinline__ void prepare(const u32x4&, int) {}
    template <class W>
    __device__ __forceinline__ void get(W& w, int, int j, int d, QsOut& o) {
        if (d == 0) w.begin(j);
        const uint32_t v = w.at(j, d) ^ 0x80808080u;  // q + 128 per byte
        o.a[2 * d] = u_of(h2_of(__builtin_amdgcn_perm(0x64646464u, v, 0x04020400u)) + h2_all(-1152.0f));
        o.a[2 * d + 1] = u_of(h2_of(__builtin_amdgcn_perm(0x64646464u, v, 0x04030401u)) + h2_all(-1152.0f));
    }
};
template <>
struct QsOperand<kQ4_0> {
    __device__ __forceinline__ void prepare(const u32x4&, int) {}
    template <class W>
    __device__ __forceinline__ void get(W& w, int g, int j, int d, QsOut& o) {
        if (d == 0) w.begin(j);
        // values 0-15 are the low nibbles of the 16 bytes, 16-31 the high ones
        const uint32_t v = w.at(j, d) >> (4 * (kgroup(g) >> 1));
        o.a[2 * d] = u_of(h2_of((v & 0x000f000fu) | 0x64006400u) + h2_all(-1032.0f));
        o.a[2 * d + 1] = u_of(h2_of(((v >> 8) & 0x000f000fu) | 0x64006400u) + h2_all(-1032.0f));
    }
};
__device__ __forceinline__ half8 h8_of(const uint32_t (&v)[4]) {
    return __builtin_bit_cast(half8, make_uint4(v[0], v[1], v[2], v[3]));
}

template <int TYPE, int TF>
__global__ __launch_bounds__(512, 1) void matbatch_qs_stream_kernel(
    MbMats mats, size_t rbytes, const _Float16* __restrict xq, const float* __restrict dxs,
    const _Float16* __restrict pq, const float* __restrict rscale, int32_t b, int32_t k, int32_t kchunk,
    float* __restrict part, int32_t xmap_tg) {
    constexpr int WAVES = 8, BM = 16 * TF, BN = kQsRows, RF = 2;
    constexpr bool SUPER = TYPE == kQ4_K || TYPE == kQ6_K;  // d per super-block, K of whole super-blocks
    constexpr int NP = TYPE == kQ6_K ? 2 : 1;               // products per block
    constexpr int OLD = BN + 4;
    constexpr int kXHalves = BM * OLD;  // a q stage, or half of the tokens' output rows as floats
    // stage s: q [token][256] with the 16-byte segments of token t at
    // positions c ^ (t % 16) (conflict-free reads of one segment by 16
    // tokens), d_x / s [token][8] with block j at j ^ (t / 4 % 4), P [token][8
    // hi, 8 lo] in 8-byte pieces swapped the same way (one piece read by 16
    // tokens hits distinct banks); separate arrays, so that a load into one
    // stage does not make the compiler wait before reads of another
    constexpr int kP = TYPE == kQ4_K ? 16 * BM : 8;
    constexpr bool S3 = TF < 8;  // three stages (two of 128 tokens fill the LDS)
    __shared__ __align__(16) _Float16 xs0[kXHalves], xs1[kXHalves], xs2[S3 ? kXHalves : 8];
    __shared__ __align__(16) float sd0[8 * BM], sd1[8 * BM], sd2[S3 ? 8 * BM : 4];
    __shared__ __align__(16) _Float16 sp0[kP], sp1[kP], sp2[S3 ? kP : 8];
    __shared__ __align__(16) float srs[BM];
    // per wave: its rows' d and dmin, or their d of each block
    __shared__ __align__(16) float sdm[WAVES][SUPER ? 2 : 8][32];

    // the work-group's row group, token group and K range.  Without a split
    // the 1-D grid can be dealt over the XCDs (work-group i runs on XCD i %
    // 8, each with its own L2): xmap > 0 (token groups, a multiple of 8):
    // each XCD keeps one eighth of the token groups and walks the row
    // groups, its concurrent work-groups sharing row groups' weights and its
    // token groups' activations; xmap < 0 (-row groups, a multiple of 8):
    // each XCD keeps one eighth of the row groups, token groups fastest, so
    // every weight is read by one XCD and the activations by all
    int bx, by, bz;
    if (xmap_tg > 0) {
        const int lin = static_cast<int>(blockIdx.x), xcd = lin & 7, slot = lin >> 3, tpx = xmap_tg / 8;
        bx = slot / tpx;
        by = xcd * tpx + slot % tpx;
        bz = 0;
    } else if (xmap_tg < 0) {
        const int lin = static_cast<int>(blockIdx.x), xcd = lin & 7, slot = lin >> 3;
        const int rgs = -xmap_tg, tgs = static_cast<int>(gridDim.x) / rgs;
        bx = xcd * (rgs / 8) + slot / tgs;
        by = slot % tgs;
        bz = 0;
    } else {
        bx = static_cast<int>(blockIdx.x);
        by = static_cast<int>(blockIdx.y);
        bz = static_cast<int>(blockIdx.z);
    }
    const uint8_t* __restrict w = mats.w[0];
    float* __restrict y = mats.y[0];
    int32_t n = mats.n[0], tile0 = 0, npre = 0;
#pragma unroll
    for (int i = 1; i < kMaxMbMats; ++i) {
        if (mats.count > i && bx >= mats.tile0[i]) {
            w = mats.w[i];
            y = mats.y[i];
            n = mats.n[i];
            tile0 = mats.tile0[i];
            npre = mats.npre[i];
        }
    }
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int l16 = lane & 15, lg = lane >> 4;
    const int32_t t0 = by * BM, n0 = (bx - tile0) * BN;
    const int32_t kb = bz * kchunk, ke = min(k, kb + kchunk);
    const int32_t nsb = (ke - kb + 255) / 256;  // super-blocks of the range
    const int32_t rows_here = min(BM, b - t0), wrows_here = min(BN, n - n0);

    // this lane's weight rows, 32 wv + 16 f + l % 16; rows past N and
    // super-blocks past the range read zeros (offsets past the resource)
    using W = QsW<TYPE, kQsWide<TYPE, TF>>;
    using H = QsH<TYPE>;
    constexpr int32_t kWB = TYPE == kQ6_K ? 210 : TYPE == kQ8_0 ? 272 : 144;  // bytes of a super-block
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(w + static_cast<size_t>(n0) * rbytes), static_cast<short>(0),
        wrows_here * static_cast<int32_t>(rbytes), 0x00020000);
    auto row_at = [&](int32_t row) {
        return row < wrows_here ? row * static_cast<int32_t>(rbytes) + kb / 256 * kWB : kMfOob / 2;
    };
    const int32_t wbase[RF] = {row_at(32 * wv + l16), row_at(32 * wv + 16 + l16)};
    const int32_t hbase = row_at(32 * wv + (lane & 31));
    struct SbRegs {
        H h;
        W f[RF];
    };
    SbRegs R;
    // part P of super-block s
    auto wload = [&]<int P>(std::integral_constant<int, P>, int32_t s) {
        const int32_t nblk = SUPER ? 8 : (ke - kb - 256 * s) / 32, at = s < nsb ? s * kWB : kMfOob / 2;
        if constexpr (P == -1) R.h.load(wrs, hbase + at);
#pragma unroll
        for (int f = 0; f < RF; ++f) R.f[f].template load<P>(wrs, wbase[f] + at, lg, nblk);
    };
    // the activations of super-block s into a stage (token rows past B and
    // values past K read zeros); with fewer than 64 tokens some waves load
    // the same d / s and P pieces again, so that every wave issues kXLoads
    constexpr int kXQ = TF, kXP = TF > 4 ? TF / 4 : 1;  // q loads, d / s and P loads per wave
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16*>(xq + static_cast<size_t>(t0) * k), static_cast<short>(0),
        rows_here * k * static_cast<int32_t>(sizeof(_Float16)), 0x00020000);
    const __amdgpu_buffer_rsrc_t drs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(dxs + static_cast<size_t>(t0) * (k / 32)), static_cast<short>(0),
        rows_here * (k / 32) * static_cast<int32_t>(sizeof(float)), 0x00020000);
    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16*>(TYPE == kQ4_K ? pq + static_cast<size_t>(t0) * (k / 256) * 16 : xq), static_cast<short>(0),
        TYPE == kQ4_K ? rows_here * (k / 256) * 16 * static_cast<int32_t>(sizeof(_Float16)) : 0, 0x00020000);
    auto xload = [&](_Float16* xst, float* sdt, _Float16* spt, int32_t s) {
        // a wave's loads differ by a wave-uniform distance (16 or 64 tokens);
        // the lane's offsets are hidden from the compiler, which would
        // otherwise keep a register for each load across the loop
        const int32_t k0 = kb + 256 * s, past = s < nsb ? 0 : kMfOob;
        const int tq = 2 * wv + (lane >> 5), c = (lane & 31) ^ (tq & 15);  // token rows 2 wv, 2 wv + 1 (+ 16 i)
        int32_t vq = (tq * k + 8 * c) * 2;
        const int pw = TF >= 4 ? wv : wv % (2 * TF);
        // tokens 8 pw .. (+ 64 i); the swizzles of d_x / s and P
        const int tp = 8 * pw + (lane >> 3), sw = (tp >> 2) & 3, blk = (lane & 7) ^ sw;
        int32_t vd = (tp * (k / 32) + blk) * 4, vp = (tp * (k / 256) * 16 + 2 * ((lane & 7) ^ (2 * sw))) * 2;
        if constexpr (!SUPER) {
            vq = k0 + 8 * c < ke ? vq : kMfOob / 2;
            vd = k0 + 32 * blk < ke ? vd : kMfOob / 2;
        }
        asm volatile("" : "+v"(vq), "+v"(vd), "+v"(vp));
#pragma unroll
        for (int i = 0; i < kXQ; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (lds_ptr)(xst + 512 * (i * WAVES + wv)), 16,
                                                     vq + (past ? kMfOob / 2 : (16 * i * k + k0) * 2), 0, 0, 0);
#pragma unroll
        for (int i = 0; i < kXP; ++i) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(drs, (lds_ptr)(sdt + 64 * (8 * i + pw)), 4,
                                                     vd + (past ? kMfOob / 2 : (64 * i * (k / 32) + k0 / 32) * 4), 0, 0,
                                                     0);
            if constexpr (TYPE == kQ4_K)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    prs, (lds_ptr)(spt + 128 * (8 * i + pw)), 4,
                    vp + (past ? kMfOob / 2 : (64 * i * (k / 256) + k0 / 256) * 32), 0, 0, 0);
        }
    };
    constexpr int kXLoads = kXQ + kXP * (TYPE == kQ4_K ? 2 : 1);
    // the loads that may be in flight past a super-block's barrier: its own
    // (weights of the next one and, with three stages, activations two ahead)
    constexpr int kLoads = H::kLoads + RF * W::kLoads + (S3 ? kXLoads : 0);
    auto wfirst = [&] {
        [&]<int... P>(std::integer_sequence<int, P...>) {
            (wload(std::integral_constant<int, P - 1>{}, 0), ...);
        }(std::make_integer_sequence<int, 9>{});
    };
    // up to 64 tokens the weights first, which come from farthest away, and
    // the row scales before them, without a branch, so that their wait covers
    // nothing else (the 128-token kernel spills 10 registers in this order:
    // 8% slower)
    if constexpr (S3) {
        const float rsv = rscale[t0 + min(tid, rows_here - 1)];
        wfirst();
        xload(xs0, sd0, sp0, 0);
        xload(xs1, sd1, sp1, 1);
        if (tid < BM) srs[tid] = rsv;
        step_barrier<kXLoads>();
    } else {
        if (tid < BM) srs[tid] = rscale[t0 + min(tid, rows_here - 1)];
        xload(xs0, sd0, sp0, 0);
        wfirst();
        step_barrier<kLoads>();
    }

    floatx4 acc[RF][TF], S[RF][TF];
#pragma unroll
    for (int f = 0; f < RF; ++f)
#pragma unroll
        for (int t = 0; t < TF; ++t) acc[f][t] = S[f][t] = floatx4{};

    // super-block s from its registers and stage, the next one's weights
    // loaded as the registers fall free
    auto process = [&](const _Float16* xst, const float* sdt, const _Float16* spt, int32_t s) {
        QsOperand<TYPE> op[RF];
        u32x4 hf[RF] = {};
        if constexpr (SUPER) spread(R.h.h, hf);
#pragma unroll
        for (int f = 0; f < RF; ++f) op[f].prepare(hf[f], lg);
        // the accumulator rows' scales, exchanged through LDS within the wave
        if constexpr (TYPE == kQ4_K) {
            if (lane < 32) {
                sdm[wv][0][lane] = half_bits_to_float(R.h.h.x & 0xffffu);
                sdm[wv][1][lane] = half_bits_to_float(R.h.h.x >> 16);
            }
        } else if constexpr (TYPE == kQ6_K) {
            if (lane < 32) sdm[wv][0][lane] = half_bits_to_float(R.h.d);
        } else {
#pragma unroll
            for (int f = 0; f < RF; ++f)
#pragma unroll
                for (int e = 0; e < 2; ++e) sdm[wv][2 * lg + e][16 * f + l16] = half_bits_to_float(R.f[f].d[e]);
        }
        wload(std::integral_constant<int, -1>{}, s + 1);
        // LDS offsets; hidden from the compiler, which would otherwise keep
        // one register per block for each across the loop
        int xa = 256 * l16 + 8 * (kgroup(lg) ^ l16), da = 8 * l16 + (l16 >> 2);
        asm volatile("" : "+v"(xa), "+v"(da));
        auto x_at = [&](int j, int t) {
            return *reinterpret_cast<const half8*>(&xst[(xa ^ (32 * j)) + 4096 * t]);
        };
        auto dx_at = [&](int j, int t) { return sdt[(da ^ j) + 128 * t]; };
        QsOut wq[2][RF];
        floatx4 dr[2][RF];
        auto dr_at = [&](int j, int f) { return *reinterpret_cast<const floatx4*>(&sdm[wv][SUPER ? 0 : j][16 * f + 4 * lg]); };
        auto mul = [&](const QsOut& o, const half8& x) {
            floatx4 v = __builtin_amdgcn_mfma_f32_16x16x32_f16(h8_of(o.a), x, floatx4{}, 0, 0, 0);
            if constexpr (NP == 2) v = __builtin_amdgcn_mfma_f32_16x16x32_f16(h8_of(o.b), x, v, 0, 0, 0);
            return v;
        };
        auto scale = [&](int j, int f, int t, float dx, const floatx4& v) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float c = SUPER ? dx : dx * dr[j & 1][f][r];
                S[f][t][r] = j == 0 ? c * v[r] : fmaf(c, v[r], S[f][t][r]);
            }
        };
#pragma unroll
        for (int f = 0; f < RF; ++f) {
            op[f].get(R.f[f], lg, 0, 0, wq[0][f]);
            op[f].get(R.f[f], lg, 0, 1, wq[0][f]);
            if constexpr (!SUPER) dr[0][f] = dr_at(0, f);
        }
        if constexpr (TF >= 4) {
            // One region per block and token tile: a region multiplies its
            // tile, scales the tile of the region before it, reads the
            // activations kAhead regions ahead and forms its share of the
            // next block's weights (a quarter every TF / 4 regions).  The
            // scheduling barriers keep that order (left alone, the compiler
            // reads and forms far ahead and spills).
            constexpr int kAhead = TYPE == kQ4_K ? 4 : 2, NX = kAhead + 1;
            half8 xo[NX];
            float dx[NX];
            floatx4 blk[2][RF];
            auto read = [&](int rg) {
                xo[rg % NX] = x_at(rg / TF, rg % TF);
                dx[rg % NX] = dx_at(rg / TF, rg % TF);
            };
            float dxp = 0.0f;
#pragma unroll
            for (int i = 0; i < kAhead; ++i) read(i);
            auto region = [&]<int rg>(std::integral_constant<int, rg>) {
                constexpr int j = rg / TF, t = rg % TF, q = t * 4 / TF;
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int f = 0; f < RF; ++f) blk[rg & 1][f] = mul(wq[j & 1][f], xo[rg % NX]);
                __builtin_amdgcn_sched_barrier(0);  // products first: their results rest until the next region
                if constexpr (rg > 0) {
#pragma unroll
                    for (int f = 0; f < RF; ++f) scale((rg - 1) / TF, f, (rg - 1) % TF, dxp, blk[(rg - 1) & 1][f]);
                }
                dxp = dx[rg % NX];
                if constexpr (rg + kAhead < 8 * TF) read(rg + kAhead);
                if constexpr (t == 0) wload(std::integral_constant<int, j>{}, s + 1);
                if constexpr (j < 7 && t % (TF / 4) == 0) {
                    op[q >> 1].get(R.f[q >> 1], lg, j + 1, q & 1, wq[(j + 1) & 1][q >> 1]);
                    if constexpr (!SUPER && q == 3) {
#pragma unroll
                        for (int f = 0; f < RF; ++f) dr[(j + 1) & 1][f] = dr_at(j + 1, f);
                    }
                }
            };
            [&]<int... G>(std::integer_sequence<int, G...>) {
                (region(std::integral_constant<int, G>{}), ...);
            }(std::make_integer_sequence<int, 8 * TF>{});
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int f = 0; f < RF; ++f) scale(7, f, TF - 1, dxp, blk[1][f]);
        } else {
            auto block = [&]<int j>(std::integral_constant<int, j>) {
                __builtin_amdgcn_sched_barrier(0);
                floatx4 blk[RF][TF];
                float dx[TF];
#pragma unroll
                for (int t = 0; t < TF; ++t) {
                    const half8 xo = x_at(j, t);
                    dx[t] = dx_at(j, t);
#pragma unroll
                    for (int f = 0; f < RF; ++f) blk[f][t] = mul(wq[j & 1][f], xo);
                }
                wload(std::integral_constant<int, j>{}, s + 1);
                if constexpr (j < 7) {
#pragma unroll
                    for (int f = 0; f < RF; ++f) {
                        op[f].get(R.f[f], lg, j + 1, 0, wq[(j + 1) & 1][f]);
                        op[f].get(R.f[f], lg, j + 1, 1, wq[(j + 1) & 1][f]);
                        if constexpr (!SUPER) dr[(j + 1) & 1][f] = dr_at(j + 1, f);
                    }
                }
#pragma unroll
                for (int t = 0; t < TF; ++t)
#pragma unroll
                    for (int f = 0; f < RF; ++f) scale(j, f, t, dx[t], blk[f][t]);
            };
            [&]<int... J>(std::integer_sequence<int, J...>) {
                (block(std::integral_constant<int, J>{}), ...);
            }(std::make_integer_sequence<int, 8>{});
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (TYPE == kQ4_K) {
            // acc += d S - dmin (m . P): the mins of sub-blocks 4 (g % 2) .. + 3
            // against P hi (g < 2) and P lo, K = 16 in one product
            half4 mo[RF];
#pragma unroll
            for (int f = 0; f < RF; ++f) {
                const uint32_t m = (lg & 1) != 0 ? op[f].mn[1] : op[f].mn[0];
                const half2 a = h2_of(__builtin_amdgcn_perm(0x64646464u, m, 0x04010400u)) + h2_all(-1024.0f);
                const half2 c = h2_of(__builtin_amdgcn_perm(0x64646464u, m, 0x04030402u)) + h2_all(-1024.0f);
                mo[f] = __builtin_shufflevector(a, c, 0, 1, 2, 3);
            }
#pragma unroll
            for (int f = 0; f < RF; ++f) {
                const floatx4 d = *reinterpret_cast<const floatx4*>(&sdm[wv][0][16 * f + 4 * lg]);
                const floatx4 dm = *reinterpret_cast<const floatx4*>(&sdm[wv][1][16 * f + 4 * lg]);
#pragma unroll
                for (int t = 0; t < TF; ++t) {
                    const half4 po = *reinterpret_cast<const half4*>(&spt[16 * (16 * t + l16) + 4 * (lg ^ (l16 >> 2))]);
                    const floatx4 M = __builtin_amdgcn_mfma_f32_16x16x16f16(mo[f], po, floatx4{}, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        acc[f][t][r] = fmaf(S[f][t][r], d[r], acc[f][t][r]);
                        acc[f][t][r] = fmaf(M[r], -dm[r], acc[f][t][r]);
                    }
                }
            }
        } else if constexpr (TYPE == kQ6_K) {
#pragma unroll
            for (int f = 0; f < RF; ++f) {
                const floatx4 d = *reinterpret_cast<const floatx4*>(&sdm[wv][0][16 * f + 4 * lg]);
#pragma unroll
                for (int t = 0; t < TF; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[f][t][r] = fmaf(S[f][t][r], d[r], acc[f][t][r]);
            }
        } else {
#pragma unroll
            for (int f = 0; f < RF; ++f)
#pragma unroll
                for (int t = 0; t < TF; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[f][t][r] += S[f][t][r];
        }
    };

    // super-block s in stage s % 3 (% 2): each starts the loads of the
    // activations two (one) ahead, into the stage the one before it left, and
    // ends with the barrier after which the next stage is in place for every
    // wave and its own may be refilled
#define GNCX_QS_STEP(XA, DA, PA, XC, DC, PC, OFF) \
    xload(XC, DC, PC, s + (OFF) + (S3 ? 2 : 1));  \
    process(XA, DA, PA, s + (OFF));               \
    step_barrier<kLoads>();                       \
    if (s + (OFF) + 1 >= nsb) break;
    if constexpr (S3) {
        for (int32_t s = 0; s < nsb; s += 3) {
            GNCX_QS_STEP(xs0, sd0, sp0, xs2, sd2, sp2, 0)
            GNCX_QS_STEP(xs1, sd1, sp1, xs0, sd0, sp0, 1)
            GNCX_QS_STEP(xs2, sd2, sp2, xs1, sd1, sp1, 2)
        }
    } else {
        for (int32_t s = 0; s < nsb; s += 2) {
            GNCX_QS_STEP(xs0, sd0, sp0, xs1, sd1, sp1, 0)
            GNCX_QS_STEP(xs1, sd1, sp1, xs0, sd0, sp0, 1)
        }
    }
#undef GNCX_QS_STEP

    // the tile as [token][BN + 4] floats in LDS, then whole token rows out;
    // first the loads past the range, which write zeros into a stage and which
    // __syncthreads() does not wait for by itself
    step_barrier<0>();
    constexpr int HT = BM / 2;  // tokens per stage array
#pragma unroll
    for (int t = 0; t < TF; ++t) {
        const int tok = 16 * t + l16;
        float* ost = reinterpret_cast<float*>(tok < HT ? xs0 : xs1) + (tok % HT) * OLD;
        const float rs = srs[tok];
#pragma unroll
        for (int f = 0; f < RF; ++f)
            *reinterpret_cast<floatx4*>(&ost[32 * wv + 16 * f + 4 * lg]) = acc[f][t] * rs;
    }
    __syncthreads();
    float* dst = gridDim.z > 1 ? part + (static_cast<size_t>(bz) * mats.ntot + npre) * b : y;
    if ((n & 3) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
        // 4 rows per lane, one token per wave and step
        const int c = 4 * lane;
        for (int t = wv; t < rows_here; t += WAVES) {
            const float* ost = reinterpret_cast<const float*>(t < HT ? xs0 : xs1) + (t % HT) * OLD;
            if (c < wrows_here)
                *reinterpret_cast<floatx4*>(&dst[static_cast<size_t>(t0 + t) * n + n0 + c]) =
                    *reinterpret_cast<const floatx4*>(&ost[c]);
        }
    } else if ((n & 1) == 0 && (reinterpret_cast<uintptr_t>(dst) & 7u) == 0) {
        const int c = 2 * (tid & 127);
#pragma unroll 4
        for (int t = tid >> 7; t < rows_here; t += 4) {
            const float* ost = reinterpret_cast<const float*>(t < HT ? xs0 : xs1) + (t % HT) * OLD;
            if (c < wrows_here)
                *reinterpret_cast<float2*>(&dst[static_cast<size_t>(t0 + t) * n + n0 + c]) =
                    *reinterpret_cast<const float2*>(&ost[c]);
        }
    } else {
        const int c = tid & 255;
#pragma unroll 4
        for (int t = tid >> 8; t < rows_here; t += 2) {
            const float* ost = reinterpret_cast<const float*>(t < HT ? xs0 : xs1) + (t % HT) * OLD;
            if (c < wrows_here) dst[static_cast<size_t>(t0 + t) * n + n0 + c] = ost[c];
        }
    }
}

// ---- BF16 weights, fp32 activations -------------------------------------------
//
// The reference multiplies fp32 activations with BF16 weights in fp32
// (cpp:1432-1461).  Here the product runs on the bf16 matrix cores without
// rounding the activations: x = h + m + l exactly, each part the top 16 bits
// of what the parts before it left (8 significant bits each, 24 in all), and
// three v_mfma_f32_16x16x32_bf16 per tile and 32-value K slice.  Every
// product of two bf16 values is exact in fp32.
//
// A work-group is 8 waves of MT 16-row weight fragments each (128 MT rows)
// times 16 NT tokens.  A weight operand is 16 bytes of one row, so the waves
// load theirs from memory straight into registers, a stage (128 of K) ahead;
// the tokens' fp32 values are loaded a stage ahead too, split on their way
// into LDS (three bf16 arrays per stage, two stages) and read from there by
// every wave.  Each stage is a sum of its own, the smaller parts first; eight
// stages add up in T and those sums in acc, so no chain of roundings at the
// full size is longer than K / 1024.  Against the 64-bit product (relative L2)
// at K = 256 / 1024 / 4096 / 14336: 0.70 / 0.80 / 0.93-1.05 / 1.07-1.28e-7;
// matbatch_rowtok_kernel 0.87 / 0.94 / 1.06 / 1.35e-7; one chain over all
// stages, folded every 256 values, 1.3-1.7e-7.
// Bound: the weight bytes up to about 64 tokens, then the three products (960
// of the 1114 bf16 TFLOP/s a large library product reaches here at 4096 x
// 4096, B = 2048).
constexpr int kBfKs = 128;  // K per stage
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// bf16 parts of 8 values: truncated top 16 bits, the remainder again, and the
// rest (exact: at most 8 significant bits are left).  Infinite or NaN values
// leave NaN in the lower parts (the output stage's check; zeros below an
// infinite value, which then needed no check, cost 2-3% on finite ones).
__device__ __forceinline__ void split3(const float (&v)[8], uint4& h, uint4& m, uint4& l) {
    uint32_t ho[4], mo[4], lo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t p[3][2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float a = v[2 * i + e];
            p[0][e] = __builtin_bit_cast(uint32_t, a);
            const float r1 = a - __builtin_bit_cast(float, p[0][e] & 0xffff0000u);
            p[1][e] = __builtin_bit_cast(uint32_t, r1);
            const float r2 = r1 - __builtin_bit_cast(float, p[1][e] & 0xffff0000u);
            p[2][e] = __builtin_bit_cast(uint32_t, r2);
        }
        ho[i] = __builtin_amdgcn_perm(p[0][1], p[0][0], 0x07060302u);
        mo[i] = __builtin_amdgcn_perm(p[1][1], p[1][0], 0x07060302u);
        lo[i] = __builtin_amdgcn_perm(p[2][1], p[2][0], 0x07060302u);
    }
    h = make_uint4(ho[0], ho[1], ho[2], ho[3]);
    m = make_uint4(mo[0], mo[1], mo[2], mo[3]);
    l = make_uint4(lo[0], lo[1], lo[2], lo[3]);
}

template <int MT, int NT>
__global__ __launch_bounds__(512, 1) void matbatch_bf16_kernel(const uint8_t* __restrict w, size_t rbytes,
                                                               const float* __restrict x, int32_t b, int32_t k,
                                                               int32_t n, int32_t kchunk, float* __restrict y,
                                                               float* __restrict part, int32_t xmap_tg) {
    constexpr int WR = 16 * MT, BN = 8 * WR, BM = 16 * NT;  // rows per wave and group, tokens
    constexpr int KS = kBfKs, NKS = KS / 32, SEGS = KS / 8;
    constexpr int XI = BM * SEGS >= 512 ? BM * SEGS / 512 : 1;  // 8-value pieces per thread and stage
    constexpr int OLD = BN + 4;                                 // floats per output row in LDS
    constexpr size_t kXBytes = size_t{2} * 3 * BM * KS * 2, kOBytes = size_t{4} * BM * OLD;
    __shared__ __align__(16) char smem[kXBytes > kOBytes ? kXBytes : kOBytes];
    // part p of stage s: [token][KS] with the 16-byte segments of token t at
    // positions c ^ (t % 16), so 16 tokens reading one segment hit distinct banks
    auto xs = [&](int s, int p) { return reinterpret_cast<uint16_t*>(smem) + (s * 3 + p) * BM * KS; };

    int bx, by, bz;
    if (xmap_tg > 0) {  // token groups dealt over the XCDs (as matbatch_qs_stream_kernel)
        const int lin = static_cast<int>(blockIdx.x), xcd = lin & 7, slot = lin >> 3, tpx = xmap_tg / 8;
        bx = slot / tpx;
        by = xcd * tpx + slot % tpx;
        bz = 0;
    } else if (xmap_tg < 0) {  // row groups
        const int lin = static_cast<int>(blockIdx.x), xcd = lin & 7, slot = lin >> 3;
        const int rgs = -xmap_tg, tgs = static_cast<int>(gridDim.x) / rgs;
        bx = xcd * (rgs / 8) + slot / tgs;
        by = slot % tgs;
        bz = 0;
    } else {
        bx = static_cast<int>(blockIdx.x);
        by = static_cast<int>(blockIdx.y);
        bz = static_cast<int>(blockIdx.z);
    }
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int l16 = lane & 15, lg = lane >> 4;
    const int32_t t0 = by * BM, n0 = bx * BN;
    const int32_t kb = bz * kchunk, ke = min(k, kb + kchunk);
    const int32_t nst = (ke - kb + KS - 1) / KS;
    const int32_t rows_here = min(BM, b - t0), wrows_here = min(BN, n - n0);

    // rows past N, tokens past B and values past the range read zeros
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(w + static_cast<size_t>(n0) * rbytes), static_cast<short>(0),
        wrows_here * static_cast<int32_t>(rbytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(x + static_cast<size_t>(t0) * k), static_cast<short>(0),
        rows_here * k * static_cast<int32_t>(sizeof(float)), 0x00020000);
    u32x4 wr[2][NKS][MT], xr[XI][2];
    auto wload = [&](u32x4 (&r)[NKS][MT], int32_t s) {
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
            const int32_t kp = kb + s * KS + 32 * ks + 8 * lg;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const int32_t row = wv * WR + 16 * i + l16;
                const int32_t off = kp < ke ? row * static_cast<int32_t>(rbytes) + 2 * kp : kMfOob;
                r[ks][i] = __builtin_amdgcn_raw_buffer_load_b128(wrs, row < wrows_here ? off : kMfOob, 0, 0);
            }
        }
    };
    auto xload = [&](int32_t s) {
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const int32_t t = (tid + 512 * i) / SEGS, kp = kb + s * KS + 8 * (tid % SEGS);
            const int32_t off = t < rows_here && kp < ke ? (t * k + kp) * static_cast<int32_t>(sizeof(float)) : kMfOob;
            xr[i][0] = __builtin_amdgcn_raw_buffer_load_b128(xrs, off, 0, 0);
            xr[i][1] = __builtin_amdgcn_raw_buffer_load_b128(xrs, off, 16, 0);
        }
    };
    auto xstore = [&](int s) {
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const int t = (tid + 512 * i) / SEGS, c = (tid % SEGS) ^ (t & 15);
            if (BM * SEGS < 512 && t >= BM) continue;
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const u32x4 q = xr[i][e >> 2];
                v[e] = __builtin_bit_cast(float, (e & 3) == 0 ? q.x : (e & 3) == 1 ? q.y : (e & 3) == 2 ? q.z : q.w);
            }
            uint4 h, m, l;
            split3(v, h, m, l);
            *reinterpret_cast<uint4*>(xs(s, 0) + t * KS + 8 * c) = h;
            *reinterpret_cast<uint4*>(xs(s, 1) + t * KS + 8 * c) = m;
            *reinterpret_cast<uint4*>(xs(s, 2) + t * KS + 8 * c) = l;
        }
    };
    floatx4 acc[MT][NT], T[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = T[i][j] = floatx4{};
    auto compute = [&](const u32x4 (&r)[NKS][MT], int s) {
        floatx4 S[MT][NT];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) S[i][j] = floatx4{};
#pragma unroll
        for (int p = 2; p >= 0; --p) {
            const uint16_t* xp = xs(s, p);
#pragma unroll
            for (int ks = 0; ks < NKS; ++ks) {
                bf16x8 xo[NT];
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    xo[j] = *reinterpret_cast<const bf16x8*>(xp + (16 * j + l16) * KS + 8 * ((4 * ks + lg) ^ l16));
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        S[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, r[ks][i]), xo[j],
                                                                         S[i][j], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) T[i][j][e] += S[i][j][e];
    };
    auto fold = [&] {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[i][j][e] += T[i][j][e];
                    T[i][j][e] = 0.0f;
                }
    };

    // stage s from register set and LDS stage s % 2: the next stage's loads
    // are issued first (x before the weights: the wait for x then leaves the
    // weights in flight), its x goes to the other LDS stage, and the barrier
    // makes it visible (step_barrier waits for no loads here)
    xload(0);
    wload(wr[0], 0);
    xstore(0);
    step_barrier<63>();
    for (int32_t s = 0; s < nst; s += 2) {
        xload(s + 1);
        wload(wr[1], s + 1);
        compute(wr[0], 0);
        if (s + 1 >= nst) break;
        xstore(1);
        step_barrier<63>();
        xload(s + 2);
        wload(wr[0], s + 2);
        compute(wr[1], 1);
        if ((s & 7) == 6) fold();
        xstore(0);
        step_barrier<63>();
    }
    fold();

    // the tile through LDS as [token][row], then whole token rows out
    __syncthreads();
    float* ost = reinterpret_cast<float*>(smem);
    int nan_out = 0;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            *reinterpret_cast<floatx4*>(&ost[(16 * j + l16) * OLD + wv * WR + 16 * i + 4 * lg]) = acc[i][j];
#pragma unroll
            for (int e = 0; e < 4; ++e) nan_out |= acc[i][j][e] != acc[i][j][e];
        }
    if (__syncthreads_or(nan_out)) {
        // A NaN output may be one of the parts alone (those of an infinite x, a
        // zero part times an infinite weight): formed again in plain fp32, a
        // wave per output.  A token or weight row found to hold a NaN
        // has NaN outputs only, and costs each wave one such sum.  (14336 ->
        // 4096 at B = 64, 50 us: one token infinite 117, all NaN 89, all infinite
        // 2410; with a lane per output 835, 7590 and 7580.)
        constexpr int CH = BN / 64;  // chunks of 64 rows; a wave takes every 8 / CH-th token of one chunk
        const int ch = wv % CH, c = 64 * ch + lane;
        uint64_t nan_rows = 0;
        for (int t = wv / CH; t < rows_here; t += 8 / CH) {
            const float v = ost[t * OLD + c];
            uint64_t todo = __ballot(v != v && c < wrows_here) & ~nan_rows;
            while (todo) {
                const int r = 64 * ch + __builtin_ctzll(todo);
                const uint8_t* wp = w + static_cast<size_t>(n0 + r) * rbytes;
                const float* xp = x + static_cast<size_t>(t0 + t) * k;
                float sum = 0.0f;
                bool wn = false, xn = false;
                for (int32_t q = kb + 8 * lane; q < ke; q += 512) {
                    const uint4 wq = *reinterpret_cast<const uint4*>(wp + 2 * static_cast<size_t>(q));
                    const float4 xa = *reinterpret_cast<const float4*>(xp + q), xb = *reinterpret_cast<const float4*>(xp + q + 4);
                    const uint32_t wd[4] = {wq.x, wq.y, wq.z, wq.w};
                    const float xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float wf = __builtin_bit_cast(float, (e & 1) == 0 ? wd[e >> 1] << 16 : wd[e >> 1] & 0xffff0000u);
                        sum += wf * xv[e];
                        wn = wn || wf != wf;
                        xn = xn || xv[e] != xv[e];
                    }
                }
                sum = wave_sum(sum);
                if (lane == 0) ost[t * OLD + r] = sum;
                if (__any(wn)) nan_rows |= todo & -todo;
                todo &= todo - 1;
                if (__any(xn)) break;
            }
        }
        __syncthreads();
    }
    float* dst = gridDim.z > 1 ? part + static_cast<size_t>(bz) * b * n : y;
    if ((n & 3) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
        constexpr int LPT = BN / 4, TPI = 512 / LPT;
        const int c = 4 * (tid % LPT);
        for (int t = tid / LPT; t < rows_here; t += TPI)
            if (c < wrows_here)
                *reinterpret_cast<floatx4*>(&dst[static_cast<size_t>(t0 + t) * n + n0 + c]) =
                    *reinterpret_cast<const floatx4*>(&ost[t * OLD + c]);
    } else {
        for (int e = tid; e < rows_here * BN; e += 512) {
            const int t = e / BN, c = e % BN;
            if (c < wrows_here) dst[static_cast<size_t>(t0 + t) * n + n0 + c] = ost[t * OLD + c];
        }
    }
}

// y = sum over the split K ranges, added in range order (deterministic);
// range z's partials are the flat block [z count, (z + 1) count).  Ranges are
// loaded U at a time, all U loads issued before the first add, without a
// branch (a range past the last reads the last again and is not added): with a
// branch around each load, 64 x 4096 outputs of 16 ranges took the call 2.6 us
// longer.  V: float, a thread per output, or floatx4 for many outputs
// (launch_reduce).
template <class V, int U>
__global__ __launch_bounds__(kThreads) void matbatch_reduce_kernel(const float* __restrict part, int32_t splits,
                                                                   RedMats r) {
    constexpr size_t W = sizeof(V) / sizeof(float);
    const size_t count = r.end[r.count - 1] / W;
    const V* __restrict p = reinterpret_cast<const V*>(part);
    const size_t i = static_cast<size_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (i >= count) return;
    V acc = p[i];
    for (int32_t z = 1; z < splits; z += U) {
        V v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = p[static_cast<size_t>(min(z + u, splits - 1)) * count + i];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (z + u < splits) acc += v[u];
    }
    float* y = r.y[0];
    size_t first = 0;
#pragma unroll
    for (int m = 1; m < kMaxMbMats; ++m) {
        if (r.count > m && i * W >= r.end[m - 1]) {
            y = r.y[m];
            first = r.end[m - 1];
        }
    }
    *reinterpret_cast<V*>(&y[i * W - first]) = acc;
}

template <class V>
void launch_reduce_t(const float* part, int32_t splits, const RedMats& r, hipStream_t stream) {
    const size_t count = r.end[r.count - 1] / (sizeof(V) / sizeof(float));
    const dim3 g(static_cast<unsigned>((count + kThreads - 1) / kThreads)), t(kThreads);
    if (splits <= 2) hipLaunchKernelGGL((matbatch_reduce_kernel<V, 1>), g, t, 0, stream, part, splits, r);
    else if (splits <= 4) hipLaunchKernelGGL((matbatch_reduce_kernel<V, 3>), g, t, 0, stream, part, splits, r);
    else if (splits <= 8) hipLaunchKernelGGL((matbatch_reduce_kernel<V, 7>), g, t, 0, stream, part, splits, r);
    else hipLaunchKernelGGL((matbatch_reduce_kernel<V, 15>), g, t, 0, stream, part, splits, r);
}

// Four outputs per thread from 1.25 * 2^20 outputs (whole, aligned groups of four),
// where the grid fills the chip either way; below that a thread each.  Whole
// calls, four / one: Q6_K K = 2048, 128 x 4096 27.3 / 21.9 us, 200 x 4096 29.4 /
// 25.2, 300 x 4096 35.8 / 33.0; Q4_K K = 4096, 64 x 4096 21.0 / 18.2, 512 x
// 2560 38.5 / 39.1, 1000 x 2048 48.7 / 49.4; Q8_0, 1000 x 2048 61.3 / 62.7.
hipError_t launch_reduce(const float* part, int32_t splits, const RedMats& r, hipStream_t stream) {
    bool four = r.end[r.count - 1] >= (size_t{5} << 18) && (reinterpret_cast<uintptr_t>(part) & 15u) == 0;
    for (int32_t i = 0; i < r.count; ++i)
        four = four && r.end[i] % 4 == 0 && (reinterpret_cast<uintptr_t>(r.y[i]) & 15u) == 0;
    if (four) launch_reduce_t<floatx4>(part, splits, r, stream);
    else launch_reduce_t<float>(part, splits, r, stream);
    return hipGetLastError();
}

// The XCD order of rg x tg work-groups with the least L2-miss traffic,
// counting each XCD's own reads of w weight and x activation bytes: by token
// groups (> 0) every XCD reads all weights and its share of the activations;
// by row groups (< 0) one XCD reads each weight and every XCD the activations
// once per round of 32 work-groups (rg tg / 256).  0: grid order.
int32_t xcd_order(int64_t rg, int64_t tg, double w, double x) {
    const double by_tok = 8.0 * w + x, by_row = w + 8.0 * x * std::max(1.0, static_cast<double>(rg * tg) / 256.0);
    if (rg % 8 == 0 && (tg % 8 != 0 || by_row < by_tok)) return -static_cast<int32_t>(rg);
    return tg % 8 == 0 ? static_cast<int32_t>(tg) : 0;
}

// A launch plan of matbatch_qs_stream_kernel: token fragments per work-group,
// K ranges and the XCD order (0: grid order)
struct QsPlan {
    int tf;
    int32_t splits, kchunk, xmap;
};

// Row groups of 256 x 16, 32, 64 or 128 tokens and K split in ranges of whole
// super-blocks, whichever is estimated fastest: rounds of 256 work-groups
// (one per CU), each a fixed part and its super-blocks, and with split K the
// reduce.  128-token tiles read each weight for twice the tokens, but pad short
// batches; tiles of 16 and 32 tokens fill the chip with fewer K ranges.
// The constants (microseconds) are fitted to whole calls of every tile and
// split at 27 shapes (B = 2 to 2048, K = 1024 to 14336, N = 512 to 40000) of
// each type: estimates within 5% in the mean, choices within 0.5% of the best
// in the mean and 5% at worst.
// n: the rows of all matrices of the launch.
QsPlan qs_plan(int32_t type, int32_t b, int32_t k, int32_t n) {
    static const double kStep[4][4] = {
        {1.8, 2.6, 3.6, 5.6},   // Q4_K
        {3.7, 4.3, 5.2, 7.9},   // Q6_K
        {6.1, 6.2, 6.2, 8.6},   // Q8_0
        {5.5, 5.8, 6.1, 8.5}};  // Q4_0
    static const double kFixed[4] = {2.3, 2.5, 3.7, 4.3};
    const double* step = kStep[type == kQ4_K ? 0 : type == kQ6_K ? 1 : type == kQ8_0 ? 2 : 3];
    const int32_t nsb = (k + 255) / 256;
    const int64_t rg = (n + kQsRows - 1) / kQsRows;
    QsPlan best{1, 1, k, 0};
    double least = 0.0;
    for (int i = 0; i < 4; ++i) {
        const int32_t tf = 1 << i;
        if (i < 2 && b > 64 * tf) continue;  // short tiles for short batches
        if (i > 0 && b <= 8 * tf) break;     // none twice as wide as the batch
        const int64_t tg = (b + 16 * tf - 1) / (16 * tf);
        // every number of ranges up to 64 that some range length gives
        for (int32_t csb = nsb;;) {
            const int32_t splits = (nsb + csb - 1) / csb;
            if (splits > 64) break;
            const double rounds = static_cast<double>((rg * tg * splits + 255) / 256);
            const double parts = static_cast<double>(splits) * b * n * 4.0;
            const double us = rounds * (kFixed[i] + csb * step[i]) + (splits > 1 ? 3.3 + parts / 2.6e6 : 0.0);
            if (least == 0.0 || us < least) {
                least = us;
                best = {tf, splits, splits > 1 ? csb * 256 : k, 0};
            }
            if (csb == 1) break;
            csb = std::min(csb - 1, (nsb + splits) / (splits + 1));
        }
    }
    if (best.splits == 1)
        best.xmap = xcd_order(rg, (b + 16 * best.tf - 1) / (16 * best.tf), static_cast<double>(n) * k * (210.0 / 256.0),
                              static_cast<double>(b) * k * 2.2);
    return best;
}

template <int TYPE, int TF>
hipError_t launch_qs_t(const MbMats& m, const QsBufs& q, int32_t b, int32_t k, const QsPlan& p, hipStream_t stream) {
    const int32_t rg = m.tile0[m.count - 1] + (m.n[m.count - 1] + kQsRows - 1) / kQsRows;
    const int32_t tg = (b + 16 * TF - 1) / (16 * TF);
    if (p.kchunk % 256 != 0 && p.splits > 1) return hipErrorInvalidValue;
    if (p.xmap > 0 && (p.xmap != tg || tg % 8 != 0 || p.splits != 1)) return hipErrorInvalidValue;
    if (p.xmap < 0 && (-p.xmap != rg || rg % 8 != 0 || p.splits != 1)) return hipErrorInvalidValue;
    const dim3 grid = p.xmap != 0 ? dim3(rg * tg) : dim3(rg, tg, p.splits);
    hipLaunchKernelGGL((matbatch_qs_stream_kernel<TYPE, TF>), grid, dim3(512), 0, stream, m, row_bytes(TYPE, k), q.xq,
                       q.dxs, q.pq, q.rscale, b, k, p.kchunk, q.part, p.xmap);
    return hipGetLastError();
}

template <int TYPE>
hipError_t launch_qs_tf(const MbMats& m, const QsBufs& q, int32_t b, int32_t k, const QsPlan& p, hipStream_t stream) {
    return p.tf == 1   ? launch_qs_t<TYPE, 1>(m, q, b, k, p, stream)
           : p.tf == 2 ? launch_qs_t<TYPE, 2>(m, q, b, k, p, stream)
           : p.tf == 4 ? launch_qs_t<TYPE, 4>(m, q, b, k, p, stream)
                       : launch_qs_t<TYPE, 8>(m, q, b, k, p, stream);
}

// The product of plan p over the matrices of m (w, y, n and count set) from
// the quantised activations in q, then with split K the reduce of the
// partials into each y
hipError_t launch_qs(int32_t type, MbMats& m, const QsBufs& q, int32_t b, int32_t k, const QsPlan& p,
                     hipStream_t stream) {
    int32_t t = 0, rows = 0;
    RedMats r{};
    for (int32_t i = 0; i < m.count; ++i) {
        m.tile0[i] = t;
        m.npre[i] = rows;
        t += (m.n[i] + kQsRows - 1) / kQsRows;
        rows += m.n[i];
        r.y[i] = m.y[i];
        r.end[i] = static_cast<size_t>(b) * rows;
    }
    m.ntot = rows;
    r.count = m.count;
    hipError_t e = hipErrorInvalidValue;
    if (type == kQ4_K) e = launch_qs_tf<kQ4_K>(m, q, b, k, p, stream);
    else if (type == kQ6_K) e = launch_qs_tf<kQ6_K>(m, q, b, k, p, stream);
    else if (type == kQ8_0) e = launch_qs_tf<kQ8_0>(m, q, b, k, p, stream);
    else if (type == kQ4_0) e = launch_qs_tf<kQ4_0>(m, q, b, k, p, stream);
    if (e != hipSuccess || p.splits == 1) return e;
    return launch_reduce(q.part, p.splits, r, stream);
}

// BF16: 256 rows per row group and 16, 32 or 64 tokens, K split in ranges of
// whole 256-value pairs of stages until about 256 work-groups run.
// Measured at 4096 x 4096, B = 64 / 100 / 512: 20.7 / 23.8 / 61.8 us; with
// about 128 work-groups 20.9 / 31.1 / 89.5, with 128 rows per row group 17.9 /
// 24.7 / 66.3 (but 50.2 against 44.5 us at 4096 x 14336, B = 64).
constexpr int kBfMT = 2;
struct BfPlan {
    int nt;
    int32_t splits, kchunk, xmap;
};
BfPlan bf16_plan(int32_t b, int32_t k, int32_t n) {
    BfPlan p{b <= 16 ? 1 : b <= 32 ? 2 : 4, 1, k, 0};
    const int32_t units = (k + 255) / 256;
    const int64_t rg = (n + 128 * kBfMT - 1) / (128 * kBfMT), tg = (b + 16 * p.nt - 1) / (16 * p.nt), wgs = rg * tg;
    int32_t splits = wgs >= 256 ? 1 : static_cast<int32_t>(256 / wgs);
    splits = std::max(1, std::min(splits, units));
    const int32_t per = (units + splits - 1) / splits;
    p.kchunk = per * 256;
    p.splits = (units + per - 1) / per;
    if (p.splits == 1) p.xmap = xcd_order(rg, tg, static_cast<double>(n) * k * 2.0, static_cast<double>(b) * k * 4.0);
    return p;
}

// The matrix kernel's fixed cost (one or two launches of long-lived
// work-groups, K split) against a wave per output: up to 4 10^7 products the
// latter.  Measured rowtok / matrix kernel: 1024 x 512 at B = 48 / 100: 6.6 /
// 12.8 and 11.7 / 13.0 us; 4096 x 4096 at B = 2 / 5: 8.4 / 11.3 and 17.2 /
// 11.3 us; 14336 x 4096 at B = 2: 38.0 / 29.0 us.
bool bf16_small(int32_t b, int32_t k, int32_t n) { return static_cast<double>(b) * k * n <= 4.0e7; }

template <int NT>
hipError_t launch_bf16_t(const uint8_t* w, const float* x, int32_t b, int32_t k, int32_t n, float* y, float* part,
                         const BfPlan& p, hipStream_t stream) {
    const int32_t rg = (n + 128 * kBfMT - 1) / (128 * kBfMT), tg = (b + 16 * NT - 1) / (16 * NT);
    const dim3 grid = p.xmap != 0 ? dim3(rg * tg) : dim3(rg, tg, p.splits);
    hipLaunchKernelGGL((matbatch_bf16_kernel<kBfMT, NT>), grid, dim3(512), 0, stream, w, row_bytes(kBF16, k), x, b, k, n,
                       p.kchunk, y, part, p.xmap);
    return hipGetLastError();
}

hipError_t launch_bf16(const uint8_t* w, const float* x, int32_t b, int32_t k, int32_t n, float* y, float* part,
                       hipStream_t stream) {
    if (bf16_small(b, k, n)) {
        hipLaunchKernelGGL(matbatch_rowtok_kernel, dim3((n + 3) / 4, b), dim3(kThreads), 0, stream, w,
                           row_bytes(kBF16, k), x, k, n, y);
        return hipGetLastError();
    }
    const BfPlan p = bf16_plan(b, k, n);
    const hipError_t e = p.nt == 1   ? launch_bf16_t<1>(w, x, b, k, n, y, part, p, stream)
                         : p.nt == 2 ? launch_bf16_t<2>(w, x, b, k, n, y, part, p, stream)
                                     : launch_bf16_t<4>(w, x, b, k, n, y, part, p, stream);
    if (e != hipSuccess || p.splits == 1) return e;
    RedMats r{};
    r.y[0] = y;
    r.end[0] = static_cast<size_t>(b) * n;
    r.count = 1;
    return launch_reduce(part, p.splits, r, stream);
}

}  // namespace

static size_t pad256(size_t v) { return (v + 255) & ~size_t{255}; }
// q [B x K] as fp16 and the blocks' d / s [B x K / 32]
static size_t xq_bytes(int32_t b, int32_t k) {
    return pad256(static_cast<size_t>(b) * k * sizeof(_Float16) + static_cast<size_t>(b) * (k / 32) * sizeof(float));
}
static size_t rscale_bytes(int32_t b) { return pad256(static_cast<size_t>(b) * sizeof(float)); }

// Q4_K: the activation sums of each 32-block as fp16 pairs [B x K/256 x 16]
static size_t pq_bytes(int32_t type, int32_t b, int32_t k) {
    return type == kQ4_K ? pad256(static_cast<size_t>(b) * (k / 256) * 16 * sizeof(_Float16)) : 0;
}

static size_t qs_bytes(int32_t type, int32_t b, int32_t k, int64_t n, int32_t splits) {
    const size_t parts = splits > 1 ? static_cast<size_t>(splits) * b * n * sizeof(float) : 0;
    return xq_bytes(b, k) + pq_bytes(type, b, k) + rscale_bytes(b) + parts + 256;
}

static QsBufs qs_bufs(void* workspace, int32_t type, int32_t b, int32_t k) {
    char* ws = static_cast<char*>(workspace);
    QsBufs q;
    q.xq = reinterpret_cast<_Float16*>(ws);
    q.dxs = reinterpret_cast<float*>(q.xq + static_cast<size_t>(b) * k);
    q.pq = type == kQ4_K ? reinterpret_cast<_Float16*>(ws + xq_bytes(b, k)) : nullptr;
    q.rscale = reinterpret_cast<float*>(ws + xq_bytes(b, k) + pq_bytes(type, b, k));
    q.part = reinterpret_cast<float*>(ws + xq_bytes(b, k) + pq_bytes(type, b, k) + rscale_bytes(b));
    return q;
}

size_t matbatch_workspace_bytes(int32_t type, int32_t b, int32_t k, int32_t n) {
    if (type == kBF16) {
        const int32_t splits = bf16_small(b, k, n) ? 1 : bf16_plan(b, k, n).splits;
        return (splits > 1 ? static_cast<size_t>(splits) * b * n * sizeof(float) : 0) + 256;
    }
    return qs_bytes(type, b, k, n, qs_plan(type, b, k, n).splits);
}

hipError_t launch_matbatch(int32_t type, const uint8_t* w, const float* x, int32_t b, int32_t k, int32_t n,
                           float* y, void* workspace, size_t workspace_bytes, hipStream_t stream, const float* up) {
    if (b <= 0 || n <= 0) return hipSuccess;
    if (k <= 0 || k > (1 << 20) || b > 65535) return hipErrorInvalidValue;  // keeps buffer offsets in int32
    if (type != kBF16 && (k % 32) != 0) return hipErrorInvalidValue;
    if ((type == kQ4_K || type == kQ6_K) && (k % 256) != 0) return hipErrorInvalidValue;
    const QsPlan p = type == kBF16 ? QsPlan{} : qs_plan(type, b, k, n);
    const size_t need = type == kBF16 ? matbatch_workspace_bytes(type, b, k, n) : qs_bytes(type, b, k, n, p.splits);
    if (workspace_bytes < need) return hipErrorInvalidValue;
    const uintptr_t wa = reinterpret_cast<uintptr_t>(w);
    if ((reinterpret_cast<uintptr_t>(x) & 15u) != 0) return hipErrorInvalidValue;
    if (type == kQ4_K || type == kBF16) {
        if ((wa & 15u) != 0 || (row_bytes(type, k) & 15u) != 0) return hipErrorInvalidValue;
    } else if ((wa & 3u) != 0) {
        return hipErrorInvalidValue;
    }
    if (type == kBF16)
        return up ? hipErrorNotSupported : launch_bf16(w, x, b, k, n, y, static_cast<float*>(workspace), stream);
    if (type != kQ4_0 && type != kQ8_0 && type != kQ4_K && type != kQ6_K) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0) return hipErrorInvalidValue;
    const QsBufs q = qs_bufs(workspace, type, b, k);
    launch_act_q(x, b, k, q, stream, up);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    MbMats m{};
    m.w[0] = w;
    m.y[0] = y;
    m.n[0] = n;
    m.count = 1;
    return launch_qs(type, m, q, b, k, p, stream);
}

namespace {

// One launch over count Q4_K matrices sharing the activation batch (and with
// split K one reduce over all of them): when every matrix is whole x-tiles of
// the plan for the summed rows (false otherwise, and the matrices go one call
// each).
bool multi_fused(int32_t type, int32_t count, const int32_t* ns, int32_t b, int32_t k, QsPlan& p, int64_t& total) {
    if (type != kQ4_K || count < 2 || count > kMaxMbMats || b <= 0 || k <= 0 || (k % 256) != 0) return false;
    total = 0;
    for (int32_t i = 0; i < count; ++i) total += ns[i];
    if (total > INT32_MAX) return false;
    for (int32_t i = 0; i < count; ++i)
        if (ns[i] % kQsRows != 0) return false;
    p = qs_plan(type, b, k, static_cast<int32_t>(total));
    return true;
}

}  // namespace

size_t matbatch_multi_workspace_bytes(int32_t type, int32_t count, const int32_t* ns, int32_t b, int32_t k) {
    QsPlan p;
    int64_t total;
    if (multi_fused(type, count, ns, b, k, p, total)) return qs_bytes(type, b, k, total, p.splits);
    size_t need = 256;
    for (int32_t i = 0; i < count; ++i) need = std::max(need, matbatch_workspace_bytes(type, b, k, ns[i]));
    return need;
}

hipError_t launch_matbatch_multi(int32_t type, int32_t count, const uint8_t* const* ws, const int32_t* ns,
                                 const float* x, int32_t b, int32_t k, float* const* ys, void* workspace,
                                 size_t workspace_bytes, hipStream_t stream) {
    if (count <= 0 || count > kMaxMbMats || !ws || !ns || !ys) return hipErrorInvalidValue;
    for (int32_t i = 0; i < count; ++i)
        if (ns[i] <= 0 || !ws[i] || !ys[i]) return hipErrorInvalidValue;
    QsPlan p;
    int64_t total;
    if (!multi_fused(type, count, ns, b, k, p, total)) {
        if (workspace_bytes < matbatch_multi_workspace_bytes(type, count, ns, b, k)) return hipErrorInvalidValue;
        for (int32_t i = 0; i < count; ++i) {
            const hipError_t e = launch_matbatch(type, ws[i], x, b, k, ns[i], ys[i], workspace, workspace_bytes, stream);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    // the checks of launch_matbatch for Q4_K
    if (workspace_bytes < qs_bytes(type, b, k, total, p.splits)) return hipErrorInvalidValue;
    if (k > (1 << 20) || b > 65535) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(x) & 15u) != 0 || (row_bytes(kQ4_K, k) & 15u) != 0) return hipErrorInvalidValue;
    for (int32_t i = 0; i < count; ++i)
        if ((reinterpret_cast<uintptr_t>(ws[i]) & 15u) != 0) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0) return hipErrorInvalidValue;
    const QsBufs q = qs_bufs(workspace, type, b, k);
    launch_act_q(x, b, k, q, stream, nullptr);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    MbMats m{};
    for (int32_t i = 0; i < count; ++i) {
        m.w[i] = ws[i];
        m.y[i] = ys[i];
        m.n[i] = ns[i];
    }
    m.count = count;
    return launch_qs(type, m, q, b, k, p, stream);
}

hipError_t launch_matbatch_multi_norm(int32_t type, int32_t count, const uint8_t* const* ws, const int32_t* ns,
                                      float* h, const float* r, const float* gamma, float eps, int32_t b, int32_t k,
                                      float* const* ys, void* workspace, size_t workspace_bytes,
                                      hipStream_t stream) {
    if (count <= 0 || count > kMaxMbMats || !ws || !ns || !ys || !h || !gamma) return hipErrorInvalidValue;
    for (int32_t i = 0; i < count; ++i)
        if (ns[i] <= 0 || !ws[i] || !ys[i]) return hipErrorInvalidValue;
    QsPlan p;
    int64_t total;
    if (!multi_fused(type, count, ns, b, k, p, total) || !norm_act_fits(h, r, gamma, k)) return hipErrorNotSupported;
    if (workspace_bytes < qs_bytes(type, b, k, total, p.splits)) return hipErrorInvalidValue;
    if (k > (1 << 20) || b > 65535 || (row_bytes(kQ4_K, k) & 15u) != 0) return hipErrorInvalidValue;
    for (int32_t i = 0; i < count; ++i)
        if ((reinterpret_cast<uintptr_t>(ws[i]) & 15u) != 0) return hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0) return hipErrorInvalidValue;
    const QsBufs q = qs_bufs(workspace, type, b, k);
    launch_norm_act_q(h, r, gamma, eps, b, k, q, stream);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    MbMats m{};
    for (int32_t i = 0; i < count; ++i) {
        m.w[i] = ws[i];
        m.y[i] = ys[i];
        m.n[i] = ns[i];
    }
    m.count = count;
    return launch_qs(type, m, q, b, k, p, stream);
}

}  // namespace gncx
