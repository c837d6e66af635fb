// gemm_rows.hip - row GEMM of a prefill chunk of 9..32 rows:
// y[m][n] = bf16(sum_k W[n][k] x[m][k]), or, SWI, bf16(silu(g) * u) of the
// gate row n and up row N + n, each rounded to bf16 first (the GEMV epilogue).
//
// MI355X design. A workgroup takes 8 or 16 W rows (SWI: 8 gate and the 8
// matching up rows) and every activation row, so that the 2048-row projections
// give every CU a workgroup; its 4 waves split K. Each wave streams its K slice through LDS
// stages of its own by direct global -> LDS loads (one instruction: 8 rows x
// 128 bytes, whole cache lines), 64 k per stage, with no workgroup barrier
// before the sums meet. Rows are stored unpadded with the 16-byte chunk c of
// row r at slot c ^ (r mod 8) (conflict-free operand reads). The slices are
// added in LDS in wave order, so the result does not depend on timing.
//
// What bounds it: the activation rows, which every workgroup reads (from L2;
// 32 rows are 4 times the bytes of its W rows), behind one memory latency.
// Per launch, weights from HBM (graph replay; the kernel before, which loaded
// 16 rows x 64 bytes per instruction straight into MFMA operands, in
// parentheses): 9 rows qkv 4.6 us (5.1), o 4.0 (5.0), gate_up + SwiGLU 11.5
// (14.0), down 7.5 (11.0); 21 rows 5.4 (6.5), 4.7 (6.5), 12.7 (17.1), 9.8
// (15.5); 32 rows 6.0 (7.5), 5.3 (7.4), 14.3 (19.1), 11.6 (18.9).
#include <hip/hip_runtime.h>

#include "bf16_math.h"
#include "error.h"
#include "mc_model.h"
#include "trace.h"

namespace mckv {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct RowsArgs {
    const uint16_t* w;
    const uint16_t* x;
    uint16_t* y;
    uint32_t ldx, ldy, M, N;
};

// Waits until at most N of this wave's global -> LDS loads are outstanding
// (they complete in order; the compiler does not track their LDS side).
template <uint32_t N>
__device__ __forceinline__ void wait_loads() {
    static_assert(N < 64u, "vmcnt is a 6-bit count");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ float round_bf16(float a) { return lo_f(pack2(a, a)); }

// X8, W8: 8-row groups of activation rows (M <= 8 X8) and W rows; K = 2048 KC in WV slices of
// 64-element steps; ST stages per wave.
template <uint32_t X8, uint32_t W8, bool SWI, uint32_t KC, uint32_t WV, uint32_t ST>
__global__ void __launch_bounds__(64u * WV) gemm_rows_kernel(const RowsArgs a) {
    constexpr uint32_t K = 2048u * KC, KW = K / WV, NS = KW / 64u;
    constexpr uint32_t LPS = X8 + W8;        // loads per stage
    constexpr uint32_t MB = (X8 + 1u) / 2u;                // 16-row MFMA blocks of x
    constexpr uint32_t kStage = LPS * 512u;                // elements
    constexpr uint32_t kRing = WV * ST * kStage, kRed = WV * MB * 64u * 8u;
    static_assert(NS >= ST && (!SWI || W8 == 2u), "whole ring in use; gate and up rows");
    __shared__ __align__(1024) uint16_t lds[kRing > kRed ? kRing : kRed];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t n0 = blockIdx.x * (SWI ? 8u : 8u * W8);
    uint16_t* ring = lds + wave * ST * kStage;
    // load i of a stage: activation rows 8 i .. 8 i + 7 (rows past M repeat row
    // M - 1, their columns are not stored), then the W rows
    const uint32_t lr = lane >> 3, chunk = 8u * ((lane & 7u) ^ lr);
    const uint16_t* src[LPS];
#pragma unroll
    for (uint32_t i = 0; i < LPS; ++i)
        src[i] = (i < X8 ? a.x + (size_t)min(8u * i + lr, a.M - 1u) * a.ldx
                         : a.w + (size_t)(n0 + (i - X8) * (SWI ? a.N : 8u) + lr) * K) +
                 wave * KW + chunk;
    auto load = [&](uint32_t s) {
#pragma unroll
        for (uint32_t i = LPS; i-- > 0u;)  // W, which comes from memory, first
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)(src[i] + 64u * s),
                (__attribute__((address_space(3))) void*)(ring + (s % ST) * kStage + i * 512u), 16,
                0, 0);
    };
#pragma unroll
    for (uint32_t s = 0; s < ST; ++s) load(s);
    f32x4_t acc[MB];
#pragma unroll
    for (uint32_t b = 0; b < MB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const uint32_t col = lane & 15u, grp = lane >> 4;
    // LDS rows of the operands: x block b, row col (its upper half repeats the
    // lower one where the last group is missing); W row col (plain: 8 rows,
    // twice; the second copy's results are not used)
    uint32_t ro[MB + 1u];
#pragma unroll
    for (uint32_t b = 0; b < MB; ++b)
        ro[b] = 64u * (16u * b + (2u * b + 1u < X8 ? col : col & 7u));
    ro[MB] = 64u * (8u * X8 + (W8 == 2u ? col : col & 7u));
#pragma unroll
    for (uint32_t s = 0; s < NS; ++s) {
        if (s + ST <= NS) wait_loads<(ST - 1u) * LPS>();
        else if (ST > 3u && s + 3u == NS) wait_loads<2u * LPS>();
        else if (ST > 2u && s + 2u == NS) wait_loads<LPS>();
        else wait_loads<0u>();
        const uint16_t* st = ring + (s % ST) * kStage;
        bf16x8_t o[2][MB + 1u];
#pragma unroll
        for (uint32_t h = 0; h < 2u; ++h)
#pragma unroll
            for (uint32_t b = 0; b <= MB; ++b)
                o[h][b] = *reinterpret_cast<const bf16x8_t*>(
                    st + ro[b] + 8u * ((4u * h + grp) ^ (col & 7u)));
        if (s + ST < NS) {
            // the operands are in registers before their stage is refilled
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            load(s + ST);
        }
#pragma unroll
        for (uint32_t h = 0; h < 2u; ++h)
#pragma unroll
            for (uint32_t b = 0; b < MB; ++b)
                acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o[h][MB], o[h][b], acc[b], 0, 0,
                                                                 0);
    }
    __syncthreads();  // every wave's loads and operand reads are done
    f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);
#pragma unroll
    for (uint32_t b = 0; b < MB; ++b) red[(wave * MB + b) * 64u + lane] = acc[b];
    __syncthreads();
    // wave b finishes activation block b; D layout: lane -> row m = col, W rows
    // 4 grp + 0..3 (8 W rows: all in grp 0 and 1; SWI: gate there, up in grp 2
    // and 3)
    constexpr uint32_t T = SWI ? 2u : 1u;
    if (wave >= MB || (grp >= 2u && (SWI || W8 == 1u))) return;
    const uint32_t m = 16u * wave + col;
    f32x4_t t[T];
#pragma unroll
    for (uint32_t r = 0; r < T; ++r) {
        t[r] = red[wave * 64u + lane + 32u * r];
#pragma unroll
        for (uint32_t v = 1; v < WV; ++v) t[r] += red[(v * MB + wave) * 64u + lane + 32u * r];
    }
    if (m >= a.M) return;
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        v[j] = SWI ? silu_mul(round_bf16(t[0][j]), round_bf16(t[T - 1u][j])) : t[0][j];
    *reinterpret_cast<uint2*>(a.y + (size_t)m * a.ldy + n0 + 4u * grp) =
        make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
}

template <uint32_t X8, uint32_t W8, bool SWI, uint32_t KC, uint32_t WV, uint32_t ST>
void launch_cfg(const RowsArgs& a, hipStream_t st) {
    hipLaunchKernelGGL((gemm_rows_kernel<X8, W8, SWI, KC, WV, ST>),
                       dim3(a.N / (SWI ? 8u : 8u * W8)), dim3(64u * WV), 0, st, a);
}
// W rows per workgroup: 8 where that gives every CU at most one (N <= 2048),
// else 16 (N = 2560, 32 rows: 5.96 us; with 8, 64 CUs have two workgroups and
// it takes 7.7). A ring of 4 stages where a CU has one workgroup, one stage
// where it has several, which then cover each other's latency (SwiGLU, 32
// rows: N = 6144 14.3 us with one stage, 15.0 with two; N = 2560 plain: 7.99
// with one, 5.96 with four; N = 512 SwiGLU, 9 rows: 7.35 with one, the kernel
// before 6.87). SwiGLU above 8192 columns streams from HBM for so long that
// bytes in flight count more than workgroups: three stages (9 / 32 rows, one
// stage, the kernel before: N = 16384 25.4 / 33.9, 26.7 / 35.8, 26.9 / 35.1;
// 65536 91.2 / 128, 96.0 / 131, 94.4 / 132; 130560 184 / 268, 189 / 271,
// 180 / 257). 8 waves were no faster anywhere.
template <uint32_t X8, bool SWI, uint32_t KC>
void launch_rows8(const RowsArgs& a, hipStream_t st) {
    constexpr uint32_t kCus = 256u;
    if constexpr (SWI) {
        if (a.N <= 8u * kCus) launch_cfg<X8, 2, true, KC, 4, 4>(a, st);
        else if (a.N <= 16u * kCus) launch_cfg<X8, 2, true, KC, 4, 2>(a, st);
        else if (a.N <= 32u * kCus) launch_cfg<X8, 2, true, KC, 4, 1>(a, st);
        else launch_cfg<X8, 2, true, KC, 4, 3>(a, st);
    } else {
        if (a.N <= 8u * kCus) launch_cfg<X8, 1, false, KC, 4, 4>(a, st);
        else if (a.N <= 16u * kCus) launch_cfg<X8, 2, false, KC, 4, 4>(a, st);
        else launch_cfg<X8, 2, false, KC, 4, 1>(a, st);
    }
}
template <bool SWI, uint32_t KC>
void launch_rows(const RowsArgs& a, hipStream_t st) {
    if (a.M <= 16u) launch_rows8<2, SWI, KC>(a, st);
    else if (a.M <= 24u) launch_rows8<3, SWI, KC>(a, st);
    else launch_rows8<4, SWI, KC>(a, st);
}

}  // namespace
}  // namespace mckv

using namespace mckv;

extern "C" mc_status_t mc_model_gemm_rows(const uint16_t* d_w, const uint16_t* d_x, uint32_t ldx,
                                          uint16_t* d_y, uint32_t ldy, uint32_t M, uint32_t N,
                                          uint32_t K, uint32_t swiglu, void* stream) {
    TraceRange trace_range("mc_model_gemm_rows");
    if (d_w == nullptr || d_x == nullptr || d_y == nullptr || M < MC_MODEL_GEMM_ROWS_MIN ||
        M > MC_MODEL_GEMM_ROWS_MAX || N == 0u || N % 16u != 0u || (K != 2048u && K != 6144u) ||
        swiglu > 1u || (swiglu && K != 2048u) || ldx < K || ldy < N || ldx % 8u != 0u ||
        ldy % 4u != 0u || (reinterpret_cast<uintptr_t>(d_w) | reinterpret_cast<uintptr_t>(d_x)) % 16u ||
        reinterpret_cast<uintptr_t>(d_y) % 8u) {
        set_error("mc_model_gemm_rows: invalid args (M=%u N=%u K=%u ldx=%u ldy=%u swiglu=%u; M "
                  "%u..%u, N a multiple of 16, K 2048 or 6144 (2048 with swiglu), ldx a "
                  "multiple of 8 and ldy of 4, w and x 16-byte and y 8-byte aligned)",
                  M, N, K, ldx, ldy, swiglu, MC_MODEL_GEMM_ROWS_MIN, MC_MODEL_GEMM_ROWS_MAX);
        return MC_E_INVALID_ARGUMENT;
    }
    hipStream_t st = (hipStream_t)stream;
    const RowsArgs a{d_w, d_x, d_y, ldx, ldy, M, N};
    if (swiglu) launch_rows<true, 1>(a, st);
    else if (K == 2048u) launch_rows<false, 1>(a, st);
    else launch_rows<false, 3>(a, st);
    return check_launch("row GEMM launch failed");
}
