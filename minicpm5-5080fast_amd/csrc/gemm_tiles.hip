// gemm_tiles.hip - the projections of a prefill chunk: y[M][N] = x[M][K] .
// W[N][K]^T (bf16 in, fp32 accumulation) on MFMA tiles, the gate_up projection
// with the SwiGLU as its epilogue, the narrow projections with K split over
// workgroups.
//
// MI355X design. A workgroup of 4 or 8 waves takes a BM x BN tile (BM
// activation rows, BN weight rows) and walks K in steps of BK = 64 or 128
// through ST LDS stages, filled by direct global -> LDS loads (16 bytes per
// lane; one wave instruction covers 8 rows x 128 bytes, whole cache lines).
// Loads with the 16 rows x 64 bytes shape of an MFMA operand reach 38 B/ns
// per CU where whole lines reach 117 (measured, L2 hits), which is why the
// operands go through LDS. Rows are stored unpadded with the 16-byte chunk c
// of row r at slot c ^ (r mod chunks), the permutation being applied to the
// global address of each lane, so both the stage's linear LDS writes and the
// MFMA operand reads (8 consecutive lanes = 8 rows, same chunk) touch every
// bank once (SQ_LDS_BANK_CONFLICT 0).
//
// Schedule: each K step's last substep starts with the wait for the next
// stage (all but ST - 2 stages of this wave's loads done), one workgroup
// barrier, and then issues the loads of stage it + ST into the stage whose
// operands are by now in registers, spread between its MFMAs so that the
// load issue never stalls the matrix cores; the next substep's operands are
// read from LDS between the same MFMAs (two register sets). 256 x 128 tile:
// 34.6 -> 31 us per 32-step round against issuing the loads in one burst.
//
// What bounds it: up to ~500 rows the bytes a CU pulls through its L1 (x and
// W tiles, about 50-80 B/ns per CU) and W's arrival from HBM (gate_up at 201
// rows: 22.1 us, 18.2 with W in cache), so the tile and split are chosen to
// give every CU one workgroup; above, the load stream and the MFMAs together,
// which overlap only in part (gate_up at 2048 rows, timing-only variants: 123
// us whole, 87 without loads, 71 with MFMAs alone, 81 without MFMAs; MFMA busy
// 57% of CU cycles there, 66% in the 256 x 256 tiles at 8448 rows, which reach
// 1.15 PFLOP/s with the SwiGLU included).
// The four projections of a layer, weights from HBM (graph replay; the library
// GEMMs that ran before and the separate SwiGLU kernel in parentheses): 64
// rows 34 us (71), 201 rows 51 (82), 512 rows 74 (97), 1024 rows 119 (139),
// 2048 rows 192 (222), 4096 rows 336 (348).
//
// Epilogues: the SwiGLU saves 12.7 us per layer at 2048 rows and 50 at 8448;
// the qkv projection's RoPE and K/V append saves the RoPE kernel and its
// launch (whole prompts: 64 tokens 2.67 -> 2.31 ms, 201 3.27 -> 2.98, 1500
// 9.4 -> 8.8, 8448 44.3 -> 44.0); its cos / sin come from a table written once
// per chunk. Loading all of a tile's cos / sin before the rotations was no
// faster than row by row.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "bf16_math.h"
#include "error.h"
#include "gemm_tiles.h"
#include "kv_internal.h"
#include "mc_model.h"
#include "trace.h"

namespace mckv {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Waits until at most N of this wave's global -> LDS loads are outstanding and
// its LDS reads have returned. The compiler does not track the LDS side of
// such loads, so every stage hand-over goes through here.
template <uint32_t N>
__device__ __forceinline__ void wait_loads() {
    static_assert(N < 64u, "vmcnt is a 6-bit count");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void load_lds16(const uint16_t* g, uint16_t* l) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                     (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}
__device__ __forceinline__ float round_bf16(float a) { return lo_f(pack2(a, a)); }

// Column (within a wave's columns) of row p of its 16-row W block b of nb.
// Blocks 2i and 2i + 1 interleave in runs of 4, so that a lane, which holds
// rows 4 grp + 0..3 of every block, has 8 adjacent columns of a block pair and
// stores 16 bytes (64-byte runs per activation row; with 8-byte stores a
// 2048-row prefill of the whole model took 11.38 ms against 11.18).
__device__ __forceinline__ uint32_t block_row(uint32_t b, uint32_t nb, uint32_t p) {
    return (b | 1u) < nb ? 32u * (b >> 1) + 8u * (p >> 2) + 4u * (b & 1u) + (p & 3u) : 16u * b + p;
}

// Pool row of the token in row m.
__device__ __forceinline__ uint16_t* rope_slot(const RopeAppend& r, uint32_t m) {
    const uint32_t pos = *r.base_pos + r.row0 + m;
    const uint32_t page = clamp_page(r.ly, r.page_table[table_index(r.ly, pos)]);
    return r.pool + token_base(r.ly, r.layer, page, pos & r.ly.pmask);
}

// grid = one workgroup per (m tile, n tile, K split). Workgroup i runs on XCD
// i mod 8: each XCD takes one contiguous range of tiles, numbered within
// groups of `group` m tiles with m fastest, so the workgroups sharing a W
// tile (and a group's x rows) meet in one L2.
// SWI: 16-row blocks of gate rows alternate with the blocks of the up rows N
// below them (w is [2N][K]); y[m][n] = bf16(silu(bf16 g) * bf16 u).
// ROPE: blocks of a head's dims 0..63 alternate with the blocks of the dims 64
// above them (a wave of one block: 8 rows of each in it); columns count dim
// pairs (N / 2), and the pair is rotated in fp32 from its bf16 projections as
// in rope_append.hip.
// Otherwise y (part == nullptr), or the fp32 sums of this K split in
// part[split][M][N].
template <uint32_t BM, uint32_t BN, uint32_t WM, uint32_t WN, uint32_t ST, uint32_t BK,
          TileEnd END>
__global__ void __launch_bounds__(64u * WM * WN)
    gemm_tile_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                     uint16_t* __restrict__ y, float* __restrict__ part, uint32_t M, uint32_t N,
                     uint32_t K, uint32_t mt, uint32_t nt, uint32_t splits, uint32_t group,
                     RopeAppend rope) {
    constexpr bool SWI = END == TileEnd::kSwiglu, ROPE = END == TileEnd::kRope;
    constexpr bool PAIR = SWI || ROPE;  // W blocks of a wave come in pairs
    constexpr uint32_t NW = WM * WN, ROWS = BM + BN;
    constexpr uint32_t CPR = BK / 8u;           // 16-byte chunks per row and stage
    constexpr uint32_t RPI = 64u / CPR;         // rows one wave load covers
    constexpr uint32_t LPW = ROWS / RPI / NW;   // loads per wave and stage
    constexpr uint32_t NS = BK / 32u;           // MFMA substeps per stage
    constexpr uint32_t TM = BM / WM, TN = BN / WN, MB = TM / 16u, NB = TN / 16u;
    static_assert(ROWS % (RPI * NW) == 0u && BM % RPI == 0u, "whole loads per wave");
    static_assert(NS % 2u == 0u, "operand register sets alternate per substep");
    constexpr bool HALVES = ROPE && NB == 1u;  // a block holds 8 pairs: lo rows, hi rows
    static_assert(!PAIR || NB % 2u == 0u || HALVES, "a wave holds both sides of a pair");
    static_assert(ST * ROWS * BK * 2u <= 160u * 1024u, "LDS");
    __shared__ __align__(1024) uint16_t lds[ST][ROWS * BK];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);

    const uint32_t total = gridDim.x, xcd = blockIdx.x & 7u;
    uint32_t t = xcd * (total >> 3) + min(xcd, total & 7u) + (blockIdx.x >> 3);
    const uint32_t sp = t % splits;
    t /= splits;
    const uint32_t gi = t / (group * nt), r = t % (group * nt);
    const uint32_t gm = min(group, mt - gi * group);  // m tiles of this group
    const uint32_t m0 = (gi * group + r % gm) * BM, n0 = r / gm * (PAIR ? BN / 2u : BN);
    const uint32_t nk = K / BK / splits, k0 = sp * nk * BK;

    // Load i of this wave fills LDS rows rr..rr + RPI - 1 (x rows, then W
    // rows); x rows past M repeat the last one (their columns are not stored).
    const uint32_t lr = lane / CPR;
    const uint16_t* base[LPW];
    uint32_t off[LPW];
#pragma unroll
    for (uint32_t i = 0; i < LPW; ++i) {
        const uint32_t rr = (i * NW + wv) * RPI;
        const uint32_t chunk = (lane % CPR) ^ ((rr + lr) & (CPR - 1u));
        if (rr < BM) {
            base[i] = x + k0;
            off[i] = min(m0 + rr + lr, M - 1u) * K + 8u * chunk;
        } else {
            const uint32_t q = rr - BM + lr;
            const uint32_t wq = q / TN, b = q % TN / 16u, p = q & 15u;  // wave, block, row
            uint32_t row;
            if constexpr (SWI)
                row = min(n0 + wq * (TN / 2u) + block_row(b >> 1, NB / 2u, p), N - 1u) +
                      ((b & 1u) ? N : 0u);
            else if constexpr (HALVES) {
                const uint32_t f = min(n0 + wq * 8u + (p & 7u), N / 2u - 1u);
                row = (f >> 6) * kD + (f & 63u) + (p >= 8u ? 64u : 0u);
            } else if constexpr (ROPE) {
                const uint32_t f =
                    min(n0 + wq * (TN / 2u) + block_row(b >> 1, NB / 2u, p), N / 2u - 1u);
                row = (f >> 6) * kD + (f & 63u) + ((b & 1u) ? 64u : 0u);
            } else row = min(n0 + wq * TN + block_row(b, NB, p), N - 1u);
            base[i] = w + k0;
            off[i] = row * K + 8u * chunk;
        }
    }
    auto load = [&](uint32_t it, uint32_t i) {
        load_lds16(base[i] + (it * BK + off[i]), &lds[it % ST][(i * NW + wv) * 512u]);
    };

    f32x4_t acc[NB][MB];
#pragma unroll
    for (uint32_t i = 0; i < NB; ++i)
#pragma unroll
        for (uint32_t j = 0; j < MB; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const uint32_t wm = wv % WM, wn = wv / WM;
    const uint32_t col = lane & 15u, grp = lane >> 4;
    const uint32_t xo = (wm * TM + col) * BK, wo = (BM + wn * TN + col) * BK;
    bf16x8_t oa[2][NB], ob[2][MB];  // W (A operand) and x (B operand) blocks
    auto read = [&](uint32_t it, uint32_t h, uint32_t set, uint32_t i) {
        const uint16_t* s = lds[it % ST];
        const uint32_t slot = 8u * ((4u * h + grp) ^ (col & (CPR - 1u)));
        if (i < NB) oa[set][i] = *reinterpret_cast<const bf16x8_t*>(s + wo + i * 16u * BK + slot);
        else
            ob[set][i - NB] =
                *reinterpret_cast<const bf16x8_t*>(s + xo + (i - NB) * 16u * BK + slot);
    };
    // waits for a stage when `after` later ones have been issued
    auto wait_stage = [&](uint32_t after) {
        if (after >= ST - 1u) wait_loads<(ST - 1u) * LPW>();
        else if (ST > 3u && after == 2u) wait_loads<2u * LPW>();
        else if (ST > 2u && after == 1u) wait_loads<LPW>();
        else wait_loads<0u>();
    };

#pragma unroll
    for (uint32_t s = 0; s < ST; ++s)
        if (s < nk) {
#pragma unroll
            for (uint32_t i = 0; i < LPW; ++i) load(s, i);
        }
    wait_stage(min(nk, ST) - 1u);
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (uint32_t i = 0; i < NB + MB; ++i) read(0u, 0u, 0u, i);

    constexpr uint32_t NM = NB * MB, RPM = (NB + MB + NM - 1u) / NM;  // reads per MFMA
    // One K step. LOAD: stage it + ST follows; LAST: no later step.
    auto step = [&](uint32_t it, auto load_c, auto last_c) {
        constexpr bool LOAD = decltype(load_c)::value, LAST = decltype(last_c)::value;
#pragma unroll
        for (uint32_t h = 0; h < NS; ++h) {
            constexpr uint32_t kLastSub = NS - 1u;
            if (h == kLastSub && !LAST) {
                // this wave's operands of stage `it` are in registers; after
                // the barrier everyone's are, and stage it + 1 is complete
                if constexpr (LOAD) wait_loads<(ST - 2u) * LPW>();
                else wait_stage(nk - 2u - it);
                __builtin_amdgcn_s_barrier();
            }
#pragma unroll
            for (uint32_t e = 0; e < NM; ++e) {
                acc[e / MB][e % MB] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    oa[h & 1u][e / MB], ob[h & 1u][e % MB], acc[e / MB][e % MB], 0, 0, 0);
                if (h < kLastSub || !LAST) {
#pragma unroll
                    for (uint32_t q = e * RPM; q < (e + 1u) * RPM && q < NB + MB; ++q)
                        read(h < kLastSub ? it : it + 1u, h < kLastSub ? h + 1u : 0u,
                             (h + 1u) & 1u, q);
                }
                if constexpr (LOAD) {
                    if (h == kLastSub) {
#pragma unroll
                        for (uint32_t i = 0; i < LPW; ++i)
                            if (i * NM / LPW == e) load(it + ST, i);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);  // keep the interleaving
            }
        }
    };
    uint32_t it = 0;
    for (; it + ST < nk; ++it) step(it, std::true_type{}, std::false_type{});
    for (; it + 1u < nk; ++it) step(it, std::false_type{}, std::false_type{});
    step(it, std::false_type{}, std::true_type{});

    // D layout: lane -> activation row col, weight rows 4 grp + 0..3
#pragma unroll
    for (uint32_t j = 0; j < MB; ++j) {
        const uint32_t m = m0 + wm * TM + 16u * j + col;
        if constexpr (HALVES) {
            // lanes < 32 hold the lower dims, the lane 32 above the dims + 64
            const uint32_t f = n0 + wn * 8u + 4u * (grp & 1u), d = f & 63u;
            const uint32_t up = grp >> 1, lo_col = (f >> 6) * kD + d;
            float lo[4], hi[4], o[4];
#pragma unroll
            for (uint32_t v = 0; v < 4u; ++v) {
                const uint32_t u = __float_as_uint(round_bf16(acc[0][j][v]));
                const auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);
                lo[v] = __uint_as_float(h[0]);
                hi[v] = __uint_as_float(h[1]);
                o[v] = up ? hi[v] : lo[v];
            }
            if (m >= M || f >= N / 2u) continue;
            uint16_t* yr = y + (size_t)m * N;
            if (lo_col < kVCol) {  // q, k: rotate
                const float2* cs = reinterpret_cast<const float2*>(yr + kKCol) + d;
#pragma unroll
                for (uint32_t v = 0; v < 4u; ++v)
                    o[v] = up ? rope_rotate(hi[v], lo[v], cs[v].x, cs[v].y, false)
                              : rope_rotate(lo[v], hi[v], cs[v].x, cs[v].y, true);
            }
            uint16_t* dst = yr + lo_col;
            if (lo_col >= kKCol) dst = rope_slot(rope, m) + (lo_col - kKCol);
            *reinterpret_cast<uint2*>(dst + 64u * up) =
                make_uint2(pack2(o[0], o[1]), pack2(o[2], o[3]));
            continue;
        }
        if (m >= M) continue;
        if constexpr (ROPE && !HALVES) {
            uint16_t* yr = y + (size_t)m * N;
            const float2* cs = reinterpret_cast<const float2*>(yr + kKCol);
            uint16_t* slot = nullptr;  // the token's page row, for k / v heads
#pragma unroll
            for (uint32_t c = 0; c < NB / 2u; c += 2u) {
                constexpr uint32_t kPairs = NB / 2u;
                const bool two = c + 1u < kPairs;
                const uint32_t f = n0 + wn * (TN / 2u) + 16u * c + (two ? 8u : 4u) * grp;
                if (f >= N / 2u) continue;
                const uint32_t d = f & 63u, lo_col = (f >> 6) * kD + d;
                float lo[8], hi[8];
#pragma unroll
                for (uint32_t i = 0; i < 8u; ++i) {
                    const uint32_t cc = i < 4u ? c : min(c + 1u, kPairs - 1u);
                    lo[i] = round_bf16(acc[2u * cc][j][i & 3u]);
                    hi[i] = round_bf16(acc[2u * cc + 1u][j][i & 3u]);
                }
                if (lo_col < kVCol) {  // q, k: rotate
#pragma unroll
                    for (uint32_t i = 0; i < 8u; ++i) {
                        if (i >= 4u && !two) break;
                        const float2 t = cs[d + i];
                        const float a = lo[i], b = hi[i];
                        lo[i] = rope_rotate(a, b, t.x, t.y, true);
                        hi[i] = rope_rotate(b, a, t.x, t.y, false);
                    }
                }
                uint16_t* o = yr + lo_col;
                if (lo_col >= kKCol) {
                    if (slot == nullptr) slot = rope_slot(rope, m);
                    o = slot + (lo_col - kKCol);
                }
                if (two) {
                    *reinterpret_cast<uint4*>(o) =
                        make_uint4(pack2(lo[0], lo[1]), pack2(lo[2], lo[3]), pack2(lo[4], lo[5]),
                                   pack2(lo[6], lo[7]));
                    *reinterpret_cast<uint4*>(o + 64) =
                        make_uint4(pack2(hi[0], hi[1]), pack2(hi[2], hi[3]), pack2(hi[4], hi[5]),
                                   pack2(hi[6], hi[7]));
                } else {
                    *reinterpret_cast<uint2*>(o) =
                        make_uint2(pack2(lo[0], lo[1]), pack2(lo[2], lo[3]));
                    *reinterpret_cast<uint2*>(o + 64) =
                        make_uint2(pack2(hi[0], hi[1]), pack2(hi[2], hi[3]));
                }
            }
            continue;
        }
        // output columns of block (pair) c: 4 values, or 8 of a block pair
        constexpr uint32_t OB = SWI ? NB / 2u : NB;
        f32x4_t o[OB];
#pragma unroll
        for (uint32_t c = 0; c < OB; ++c) {
            if constexpr (SWI) {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    o[c][v] = silu_mul(round_bf16(acc[2u * c][j][v]),
                                       round_bf16(acc[2u * c + 1u][j][v]));
            } else {
                o[c] = acc[c][j];
            }
        }
        const uint32_t nw = n0 + wn * (TN / (SWI ? 2u : 1u));  // the wave's first column
#pragma unroll
        for (uint32_t c = 0; c < OB; c += 2u) {
            const bool pair = c + 1u < OB;
            const uint32_t n = nw + 16u * c + (pair ? 8u : 4u) * grp;
            if (n >= N) continue;
            const size_t e = (size_t)m * N + n;
            const f32x4_t a = o[c], b = o[pair ? c + 1u : c];
            if (!SWI && part != nullptr) {
                float* d = part + (size_t)sp * M * N + e;
                *reinterpret_cast<f32x4_t*>(d) = a;
                if (pair) *reinterpret_cast<f32x4_t*>(d + 4) = b;
            } else if (pair) {
                *reinterpret_cast<uint4*>(y + e) = make_uint4(
                    pack2(a[0], a[1]), pack2(a[2], a[3]), pack2(b[0], b[1]), pack2(b[2], b[3]));
            } else {
                *reinterpret_cast<uint2*>(y + e) =
                    make_uint2(pack2(a[0], a[1]), pack2(a[2], a[3]));
            }
        }
    }
}

template <uint32_t BM, uint32_t BN, uint32_t WM, uint32_t WN, uint32_t ST, uint32_t BK,
          TileEnd END>
void launch_tile(const GemmTiles& g, uint32_t splits, hipStream_t st) {
    constexpr uint32_t cols = END == TileEnd::kSwiglu ? BN / 2u : BN;
    const uint32_t mt = (g.M + BM - 1u) / BM, nt = (g.N + cols - 1u) / cols;
    // m tiles of about 512 rows share the W tiles of an XCD's L2
    constexpr uint32_t group = BM >= 256u ? 2u : 512u / BM;
    hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WM, WN, ST, BK, END>), dim3(mt * nt * splits),
                       dim3(64u * WM * WN), 0, st, g.x, g.w, g.y, g.part, g.M, g.N, g.K, mt, nt,
                       splits, group, g.rope);
}

// Tile shapes and their measured cost in us: a launch of r rounds of 256
// workgroups (one per CU) with n 64-element K steps each takes about
// launch + r (round + n step). Least-squares fits over 33..8448 rows of the
// model's four projections, splits 1..8, weights from HBM (residuals 4-12%
// rms; with the SwiGLU, K = 2048 only, the step holds the round's part).
// step grows with BM + BN, the bytes a K step brings in, so a larger tile does
// more per byte but leaves CUs idle when the shape gives it few tiles or a
// short last round: the plan takes the shapes and split of least estimated
// time (on the measured tables of the plain and SwiGLU forms 1.5% above the best
// choice on average, 15% at worst). The RoPE form has no fit of its own: it is
// planned with the plain form's costs, which are 7-20% under its launches (30.3
// us for 25.9 estimated at 2048 rows, 88 for 76 at 8448) but order the shapes
// alike: over 29 row counts from 33 to 8448 the planned launch is within 2% of
// the best single shape.
struct TileCost {
    float launch, round, step;  // step 0: the shape does not take this form
};
struct TileShape {
    uint16_t bm, bn, bk;
    bool rope;  // waves hold one W block, or blocks in pairs: takes the rope form
    TileCost plain, swiglu;
};
constexpr TileShape kShapes[] = {
    {32, 64, 128, true, {3.92f, 0.00f, 0.166f}, {}},
    {48, 64, 128, true, {2.46f, 1.52f, 0.190f}, {}},
    {64, 64, 128, true, {2.54f, 1.78f, 0.215f}, {}},
    {64, 64, 64, false, {}, {9.06f, 0.00f, 0.195f}},
    {64, 96, 64, false, {}, {9.17f, 0.00f, 0.255f}},
    {96, 64, 64, true, {3.89f, 0.76f, 0.243f}, {8.89f, 0.00f, 0.238f}},
    {128, 64, 64, true, {2.71f, 2.67f, 0.290f}, {6.72f, 0.00f, 0.361f}},
    {128, 96, 64, true, {2.57f, 3.47f, 0.357f}, {5.71f, 0.00f, 0.486f}},
    {128, 128, 64, true, {2.96f, 4.18f, 0.420f}, {4.95f, 0.00f, 0.562f}},
    {128, 192, 64, false, {}, {0.77f, 0.00f, 0.885f}},
    {192, 128, 64, true, {2.62f, 5.32f, 0.562f}, {0.25f, 0.00f, 0.809f}},
    {256, 128, 64, true, {3.28f, 6.54f, 0.662f}, {0.00f, 0.00f, 0.996f}},
    {160, 256, 64, true, {3.23f, 8.34f, 0.866f}, {0.00f, 0.00f, 1.318f}},
    {192, 192, 64, true, {2.73f, 7.69f, 0.785f}, {0.00f, 0.00f, 1.203f}},
    {256, 160, 64, false, {3.05f, 8.21f, 0.864f}, {}},
    {256, 192, 64, true, {5.09f, 7.37f, 0.884f}, {0.00f, 0.00f, 1.463f}},
    {192, 256, 64, true, {6.27f, 6.11f, 0.908f}, {1.67f, 0.00f, 1.402f}},
    {256, 256, 64, true, {9.61f, 4.30f, 1.116f}, {0.00f, 0.00f, 1.774f}},
};
constexpr uint32_t kShapeCount = sizeof(kShapes) / sizeof(kShapes[0]);
static_assert(kShapeCount == MC_MODEL_GEMM_TILES_SHAPES, "header constant");
constexpr uint32_t kSplits[] = {1, 2, 3, 4, 5, 6, 7, 8};
constexpr uint32_t kRound = 256u;  // CUs

const TileCost& cost_of(const TileShape& s, TileEnd end) {
    return end == TileEnd::kSwiglu ? s.swiglu : s.plain;
}
bool shape_fits(const TileShape& s, uint32_t K, TileEnd end, uint32_t splits) {
    return cost_of(s, end).step > 0.f && (end != TileEnd::kRope || s.rope) &&
           K % (s.bk * splits) == 0u;
}

}  // namespace

namespace {

// n tiles of a shape (the last one may be part empty)
uint32_t n_tiles(const TileShape& s, uint32_t N, TileEnd end) {
    const uint32_t cols = end == TileEnd::kSwiglu ? s.bn / 2u : s.bn;
    return (N + cols - 1u) / cols;
}

float estimate_us(const TileShape& s, uint32_t M, uint32_t N, uint32_t K, TileEnd end,
                  uint32_t splits) {
    const TileCost& c = cost_of(s, end);
    const uint32_t tiles = (M + s.bm - 1u) / s.bm * n_tiles(s, N, end) * splits;
    const uint32_t rounds = (tiles + kRound - 1u) / kRound;
    const float us = c.launch + (float)rounds * (c.round + (float)(K / 64u / splits) * c.step);
    // the consumer reads `splits` fp32 sums instead of one bf16 value
    return splits == 1u ? us : us + 0.3f + (float)splits * (float)M * (float)N * 1e-6f;
}

// Best shape and split for M rows in one launch; *us its estimate (shape
// kShapeCount when none fits).
void best_single(uint32_t M, uint32_t N, uint32_t K, TileEnd end, uint32_t min_splits,
                 uint32_t max_splits, uint32_t* shape, uint32_t* splits, float* us) {
    *shape = kShapeCount;
    *splits = min_splits;
    *us = 0.f;
    for (uint32_t i = 0; i < kShapeCount; ++i)
        for (const uint32_t sp : kSplits) {
            if (sp < min_splits || sp > max_splits || (sp > 1u && end != TileEnd::kPlain) ||
                !shape_fits(kShapes[i], K, end, sp))
                continue;
            const float t = estimate_us(kShapes[i], M, N, K, end, sp);
            if (*shape == kShapeCount || t < *us) {
                *shape = i;
                *splits = sp;
                *us = t;
            }
        }
}

}  // namespace

GemmPlan gemm_tiles_plan(uint32_t M, uint32_t N, uint32_t K, TileEnd end, uint32_t min_splits,
                         uint32_t max_splits, float* us_out) {
    GemmPlan p;
    float us;
    best_single(M, N, K, end, min_splits, max_splits, &p.shape0, &p.splits, &us);
    p.rows0 = M;
    if (us_out != nullptr) *us_out = us;
    if (min_splits > 1u) return p;
    // Two launches: whole rounds of a large tile over the first rows, the
    // rest on the tile that suits it, where one shape would leave most of its
    // last round's CUs idle (8448 rows of gate_up: 6 rounds of 256 x 256 and
    // 256 rows, 334 + 24 us in place of 368).
    for (uint32_t i = 0; i < kShapeCount; ++i) {
        if (!shape_fits(kShapes[i], K, end, 1u)) continue;
        const uint32_t nt = n_tiles(kShapes[i], N, end);
        for (uint32_t r = 1u; r <= 16u; ++r) {
            const uint32_t rows = kRound * r / nt * kShapes[i].bm;
            if (rows == 0u) continue;
            if (rows >= M) break;
            uint32_t shape, splits;
            float rest;
            best_single(M - rows, N, K, end, 1u, 1u, &shape, &splits, &rest);
            const float t = estimate_us(kShapes[i], rows, N, K, end, 1u) + rest + 2.f;
            if (t < us) {
                us = t;
                p = {rows, i, shape, 1u};
            }
        }
    }
    if (us_out != nullptr) *us_out = us;
    return p;
}

bool gemm_tiles_fits(uint32_t shape, uint32_t K, TileEnd end, uint32_t splits) {
    return shape < kShapeCount && splits >= 1u && splits <= 8u &&
           (end == TileEnd::kPlain || splits == 1u) && shape_fits(kShapes[shape], K, end, splits);
}

namespace {

mc_status_t launch_shape(const GemmTiles& g, uint32_t shape, uint32_t splits, hipStream_t st) {
    // one case per row of kShapes: waves over m x n, LDS stages
#define MC_TILE_END(i, WM, WN, ST, E, HAS)                                               \
    if constexpr (HAS)                                                                   \
        if (end == E)                                                                    \
            launch_tile<kShapes[i].bm, kShapes[i].bn, WM, WN, ST, kShapes[i].bk, E>(     \
                g, splits, st);
#define MC_TILE(i, WM, WN, ST)                                                           \
    case i:                                                                              \
        MC_TILE_END(i, WM, WN, ST, TileEnd::kPlain, kShapes[i].plain.step > 0.f)         \
        MC_TILE_END(i, WM, WN, ST, TileEnd::kSwiglu, kShapes[i].swiglu.step > 0.f)       \
        MC_TILE_END(i, WM, WN, ST, TileEnd::kRope, kShapes[i].rope)                      \
        break;
    const TileEnd end = g.swiglu                         ? TileEnd::kSwiglu
                        : g.rope.page_table != nullptr ? TileEnd::kRope
                                                       : TileEnd::kPlain;
    switch (shape) {
        MC_TILE(0, 1, 4, 3)
        MC_TILE(1, 1, 4, 4)
        MC_TILE(2, 2, 4, 4)
        MC_TILE(3, 2, 2, 4)
        MC_TILE(4, 4, 1, 4)
        MC_TILE(5, 2, 2, 4)
        MC_TILE(6, 4, 2, 4)
        MC_TILE(7, 4, 1, 4)
        MC_TILE(8, 2, 4, 4)
        MC_TILE(9, 2, 2, 3)
        MC_TILE(10, 2, 4, 3)
        MC_TILE(11, 4, 2, 3)
        MC_TILE(12, 2, 2, 3)
        MC_TILE(13, 2, 2, 3)
        MC_TILE(14, 2, 2, 3)
        MC_TILE(15, 4, 2, 2)
        MC_TILE(16, 2, 4, 2)
        MC_TILE(17, 2, 4, 2)
        default:
            set_error("prefill GEMM: no tile shape for %u x %u x %u", g.M, g.N, g.K);
            return MC_E_INTERNAL;
    }
#undef MC_TILE
#undef MC_TILE_END
    return check_launch("tile GEMM launch failed");
}

}  // namespace

mc_status_t gemm_tiles(const GemmTiles& g, const GemmPlan& p, hipStream_t st) {
    GemmTiles a = g;
    a.M = p.rows0;
    const mc_status_t r = launch_shape(a, p.shape0, p.splits, st);
    if (r != MC_OK || p.rows0 == g.M) return r;
    a.x += (size_t)p.rows0 * g.K;
    if (g.part != nullptr) a.part += (size_t)p.rows0 * g.N;
    else a.y += (size_t)p.rows0 * g.N;
    a.M = g.M - p.rows0;
    a.rope.row0 += p.rows0;
    return launch_shape(a, p.shape1, 1u, st);
}

}  // namespace mckv

using namespace mckv;

extern "C" mc_status_t mc_model_gemm_tiles(const uint16_t* d_w, const uint16_t* d_x,
                                           uint16_t* d_y, float* d_partials, uint32_t M,
                                           uint32_t N, uint32_t K, uint32_t swiglu,
                                           uint32_t splits, uint32_t shape, void* stream) {
    TraceRange trace_range("mc_model_gemm_tiles");
    const bool addr_ok =
        ((reinterpret_cast<uintptr_t>(d_w) | reinterpret_cast<uintptr_t>(d_x) |
          reinterpret_cast<uintptr_t>(d_partials)) % 16u) == 0u &&
        reinterpret_cast<uintptr_t>(d_y) % 16u == 0u;
    if (d_w == nullptr || d_x == nullptr || (d_y == nullptr) == (d_partials == nullptr) ||
        !addr_ok || M == 0u || M > 65535u || N == 0u || N > 65536u || N % 64u != 0u || K == 0u ||
        K > 16384u || K % 128u != 0u || swiglu > 1u || (swiglu && d_partials != nullptr) ||
        splits < 1u || splits > 8u || (splits > 1u && d_partials == nullptr) ||
        K % (128u * splits) != 0u) {
        set_error("mc_model_gemm_tiles: invalid args (M=%u N=%u K=%u swiglu=%u splits=%u; N a "
                  "multiple of 64, K of 128 x splits, exactly one of y / partials, partials for "
                  "splits > 1 and not with swiglu, 16-byte aligned pointers)",
                  M, N, K, swiglu, splits);
        return MC_E_INVALID_ARGUMENT;
    }
    const TileEnd end = swiglu ? TileEnd::kSwiglu : TileEnd::kPlain;
    GemmPlan p{M, shape, 0u, splits};
    if (shape == MC_MODEL_GEMM_TILES_AUTO) {
        p = gemm_tiles_plan(M, N, K, end, splits, splits);
    } else if (!gemm_tiles_fits(shape, K, end, splits)) {
        set_error("mc_model_gemm_tiles: shape %u does not take N=%u K=%u swiglu=%u splits=%u",
                  shape, N, K, swiglu, splits);
        return MC_E_INVALID_ARGUMENT;
    }
    GemmTiles g{d_x, d_w, d_y, d_partials, M, N, K, swiglu != 0u};
    return gemm_tiles(g, p, (hipStream_t)stream);
}

extern "C" mc_status_t mc_model_gemm_tiles_rope(const uint16_t* d_w, const uint16_t* d_x,
                                                uint16_t* d_qkv, uint32_t M, uint32_t K,
                                                const uint32_t* d_base_pos, uint32_t layer,
                                                const uint32_t* d_page_table,
                                                uint16_t* d_kv_pool, mc_kv_layout_t layout,
                                                uint32_t shape, void* stream) {
    TraceRange trace_range("mc_model_gemm_tiles_rope");
    const bool addr_ok =
        ((reinterpret_cast<uintptr_t>(d_w) | reinterpret_cast<uintptr_t>(d_x) |
          reinterpret_cast<uintptr_t>(d_qkv) | reinterpret_cast<uintptr_t>(d_kv_pool)) %
         16u) == 0u;
    RopeAppend rope{d_base_pos, d_page_table, d_kv_pool, {}, layer, 0u};
    if (d_w == nullptr || d_x == nullptr || d_qkv == nullptr || d_base_pos == nullptr ||
        d_page_table == nullptr || d_kv_pool == nullptr || !addr_ok || M == 0u || M > 65535u ||
        K == 0u || K > 16384u || K % 128u != 0u || !layout_valid(layout, &rope.ly) ||
        layer >= layout.num_layers) {
        set_error("mc_model_gemm_tiles_rope: invalid args (M=%u K=%u layer=%u; K a multiple of "
                  "128, 16-byte aligned pointers)", M, K, layer);
        return MC_E_INVALID_ARGUMENT;
    }
    GemmPlan p{M, shape, 0u, 1u};
    if (shape == MC_MODEL_GEMM_TILES_AUTO) {
        p = gemm_tiles_plan(M, kRow, K, TileEnd::kRope, 1u, 1u);
    } else if (!gemm_tiles_fits(shape, K, TileEnd::kRope, 1u)) {
        set_error("mc_model_gemm_tiles_rope: shape %u does not take K=%u", shape, K);
        return MC_E_INVALID_ARGUMENT;
    }
    return gemm_tiles({d_x, d_w, d_qkv, nullptr, M, kRow, K, false, rope}, p,
                      (hipStream_t)stream);
}

extern "C" mc_status_t mc_model_debug_gemm_tiles_plan(uint32_t M, uint32_t N, uint32_t K,
                                                      uint32_t form, uint32_t min_splits,
                                                      uint32_t max_splits, uint32_t plan[4]) {
    if (plan == nullptr || M == 0u || M > 65535u || N == 0u || N > 65536u || N % 64u != 0u ||
        K == 0u || K > 16384u || form > 2u || (form == 2u && N != kRow) || min_splits < 1u ||
        min_splits > max_splits || max_splits > 8u || (form != 0u && max_splits > 1u) ||
        K % (128u * min_splits) != 0u) {
        set_error("mc_model_debug_gemm_tiles_plan: invalid args (M=%u N=%u K=%u form=%u "
                  "splits=%u..%u)", M, N, K, form, min_splits, max_splits);
        return MC_E_INVALID_ARGUMENT;
    }
    const GemmPlan p = gemm_tiles_plan(M, N, K, (TileEnd)form, min_splits, max_splits);
    plan[0] = p.rows0;
    plan[1] = p.shape0;
    plan[2] = p.shape1;
    plan[3] = p.splits;
    return MC_OK;
}
