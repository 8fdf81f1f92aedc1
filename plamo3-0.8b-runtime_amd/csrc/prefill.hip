// Prefill kernels for gfx950: MFMA BF16 GEMM (plain or .p12 weights) with fused epilogues,
// row RMSNorm / residual kernels and the K/V cache writer.
//
//   gemm_dma_kernel Y[t][m] = sum_k X[t][k] W[m][k] for plain BF16 weights and many tokens:
//                   large tiles, operands loaded straight into swizzled LDS stages,
//                   v_mfma_f32_32x32x16_bf16, XCD-grouped tiles.
//   gemm_small_kernel  the same for fewer tokens: tiles of 16x16 blocks down to one block, so
//                   that short prompts fill the chip too.
//   gemm_kernel     the same product for .p12 weights, expanded in registers on the way to a
//                   double-buffered LDS tile.  Both replace `matrix` (Kernels.metal:149-200)
//                   for the projections and `swiglu` (Kernels.metal:202-210) as an epilogue.
//   rows_norm       `norm` (Kernels.metal:46-90) for T rows: embedding gather + norm, or
//                   post-norm + residual + next norm.
//   qk_prep         `qkv` (Kernels.metal:223-259) for a chunk: q/k RMSNorm, RoPE, K/V to
//                   cache slot pos % capacity, normalised rotated queries as BF16.
//   flash_prefill   prefill attention (Runtime.swift:389-444) as MFMA flash attention.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "device.h"
#include "kernels.h"
#include "prefill.h"

namespace plamo {
using namespace dev;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int BK = 64, LDS_STRIDE = BK + 8;  // +16 B per row against bank conflicts

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) {
    bf16x8 r;
    __builtin_memcpy(&r, &v, 16);
    return r;
}

// Weight row feeding LDS row r of a B tile.  SwiGLU tiles interleave 32 gate and 32 up rows
// (g0-31, u0-31, g32-63, u32-63, ...) so that each wave's column tiles pair gate with up.
template <int EPI>
__device__ __forceinline__ int b_row(int n0, int r) {
    if constexpr (EPI == GEMM_SWIGLU) return ((r >> 5) & 1 ? INTER : 0) + n0 + (r >> 6) * 32 + (r & 31);
    else return n0 + r;
}

// One K step of operands in registers: thread tid loads 16 bytes of rows tid/8 + 32*i.
template <int BT, int BW, int NT>
struct GemmStage {
    static constexpr int RP = NT / 8;  // rows covered by one pass of the workgroup
    uint4 a[BT / RP], b[BW / RP];
};

// Operand views of one GEMM: rows past `tokens` (activations) or `m` (plain weights) read as
// zero.  .p12 payload offsets come from the validated block table.
struct GemmViews {
    __amdgpu_buffer_rsrc_t x, w, table;
};

__device__ __forceinline__ GemmViews gemm_views(const GemmParams& p, bool packed) {
    GemmViews v;
    v.x = buffer_view(p.x, uint32_t(p.tokens) * uint32_t(p.k) * 2u);
    v.w = buffer_view(p.w, packed ? 0x7fffffffu : uint32_t(p.m) * uint32_t(p.k) * 2u);
    v.table = buffer_view(p.table, packed ? uint32_t(p.m) * uint32_t(p.k / 128) * 4u : 0u);
    return v;
}

// Loads K step k0 of both operands.  A step past the end (live == false) is still issued, with
// every offset outside its view: it reads zeros without touching memory, and the loads stay
// unconditional, so the wait before each LDS store counts only the loads of the step it stores.
template <bool PACKED, int EPI, int BT, int BW, int NT>
__device__ __forceinline__ void gemm_load(const GemmParams& p, const GemmViews& v, int t0, int n0, int k0, bool live,
                                          GemmStage<BT, BW, NT>& g) {
    constexpr int RP = GemmStage<BT, BW, NT>::RP;
    const int tid = threadIdx.x, c8 = tid & 7;
    const uint32_t K = uint32_t(p.k);
    const uint32_t kk = uint32_t(k0 + c8 * 8);
    const uint32_t kill = live ? 0u : OOB_OFFSET;
#pragma unroll
    for (int i = 0; i < BT / RP; ++i) {
        const uint32_t t = uint32_t(t0 + (tid >> 3) + RP * i);
        g.a[i] = buffer_prefetch16(v.x, ((t * K + kk) * 2u) | kill);
    }
#pragma unroll
    for (int i = 0; i < BW / RP; ++i) {
        const uint32_t row = uint32_t(b_row<EPI>(n0, (tid >> 3) + RP * i));
        if constexpr (!PACKED) {
            g.b[i] = buffer_prefetch16(v.w, ((row * K + kk) * 2u) | kill);
        } else {
            const uint32_t entry = buffer_load4(v.table, ((row * (K / 128) + kk / 128) * 4u) | kill);
            const uint32_t blk = (entry & ~63u) | kill, tag = entry & 63u;
            const uint32_t sub = (kk % 128) / 8;
            if (tag == 0) g.b[i] = buffer_load16(v.w, blk + sub * 16);
            else g.b[i] = p12_decode8(buffer_load8(v.w, blk + sub * 8), buffer_load4(v.w, blk + 128 + sub * 4), tag);
        }
    }
}

template <int BT, int BW, int NT>
__device__ __forceinline__ void gemm_store(const GemmStage<BT, BW, NT>& g, uint16_t* As, uint16_t* Bs) {
    constexpr int RP = GemmStage<BT, BW, NT>::RP;
    const int tid = threadIdx.x, c8 = tid & 7;
#pragma unroll
    for (int i = 0; i < BT / RP; ++i)
        *reinterpret_cast<uint4*>(&As[((tid >> 3) + RP * i) * LDS_STRIDE + c8 * 8]) = g.a[i];
#pragma unroll
    for (int i = 0; i < BW / RP; ++i)
        *reinterpret_cast<uint4*>(&Bs[((tid >> 3) + RP * i) * LDS_STRIDE + c8 * 8]) = g.b[i];
}

// Writes a wave's TT x TW accumulator tiles (tokens from tw0, LDS weight-row tiles of wave
// column ww) with the chosen epilogue.
template <int EPI, int TT, int TW>
__device__ __forceinline__ void gemm_epilogue(const GemmParams& p, const floatx16 (&acc)[TT][TW], int tw0, int n0, int ww,
                                              int lane) {
    // C layout of a 32x32 tile: column j = lane%32, row i = (r/4)*8 + (lane/32)*4 + r%4.
    // Stores go through views bounded by the output size, so rows past `tokens` are dropped
    // without branches (columns past m get an offset outside the view).
    const int jc = lane & 31;
    const uint32_t M = uint32_t(p.m);
    const __amdgpu_buffer_rsrc_t yv =
        EPI == GEMM_SWIGLU ? buffer_view(p.y16, uint32_t(p.tokens) * INTER * 2u)
                           : (EPI == GEMM_BF16 ? buffer_view(p.y16, uint32_t(p.tokens) * M * 2u)
                                               : buffer_view(p.y, uint32_t(p.tokens) * M * 4u));
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t t = uint32_t(tw0 + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3));
            if constexpr (EPI == GEMM_SWIGLU) {
#pragma unroll
                for (int j = 0; j < TW; j += 2) {  // LDS rows of tile j are gate rows, of j + 1 the matching up rows
                    const uint32_t m = uint32_t(n0 + ((ww * TW + j) >> 1) * 32 + jc);
                    // g / (1 + exp(-g)) with IEEE division (Kernels.metal:202-210), the exp of
                    // the decode epilogue (`exp_det`): decode and prefill round alike
                    const float gt = roundbf(acc[i][j][r]);
                    const float up = roundbf(acc[i][j + 1][r]);
                    const float silu = gt / (1.0f + exp_det(-gt));
                    buffer_store2(yv, (t * INTER + m) * 2u, uint16_t(bits(roundbf(silu) * up)));
                }
            } else {
#pragma unroll
                for (int j = 0; j < TW; ++j) {
                    const uint32_t m = uint32_t(n0 + ww * TW * 32 + j * 32 + jc);
                    const uint32_t e = m < M ? t * M + m : OOB_OFFSET / 4;
                    if constexpr (EPI == GEMM_F32) buffer_store4(yv, e * 4u, __float_as_uint(roundbf(acc[i][j][r])));
                    else if constexpr (EPI == GEMM_RAW) buffer_store4(yv, e * 4u, __float_as_uint(acc[i][j][r]));
                    else buffer_store2(yv, e * 2u, uint16_t(bits(acc[i][j][r])));
                }
            }
        }
}

// Y[t][m] = sum_k X[t][k] W[m][k] on BT x BW tiles (tokens x weight rows): four waves in a
// WT x (4 / WT) grid, each owning (BT / WT) x (BW * WT / 4) outputs as 32x32 MFMA tiles.  The
// next two K steps are in flight in registers while the current one is multiplied from LDS
// (double-buffered, one barrier per step).  Tiles are dealt to workgroups so that each XCD
// (workgroup id % 8) owns a contiguous run of tiles sharing weight columns, which keeps the
// weight tiles in that XCD's L2.  Larger tiles read fewer operand bytes per FLOP from L2.
template <bool PACKED, int EPI, int BT, int BW, int WT, int NT>
__global__ __launch_bounds__(NT) void gemm_kernel(const GemmParams p, int col_tiles, int row_tiles) {
    constexpr int WW = NT / 64 / WT, TT = BT / WT / 32, TW = BW / WW / 32;
    static_assert(EPI != GEMM_SWIGLU || TW % 2 == 0, "SwiGLU pairs gate and up tiles inside a wave");
    __shared__ __align__(16) uint16_t As[2][BT * LDS_STRIDE];
    __shared__ __align__(16) uint16_t Bs[2][BW * LDS_STRIDE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform (scalar)
    const int wt = wave / WW, ww = wave % WW;
    const int tiles = col_tiles * row_tiles;
    const int per = (tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int ct = tile / row_tiles, rt = tile % row_tiles;
    const int t0 = rt * BT;
    const int n0 = ct * (EPI == GEMM_SWIGLU ? BW / 2 : BW);
    const int nk = p.k / BK;

    floatx16 acc[TT][TW];
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < TW; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // Two K steps of operands are in flight in registers while one is multiplied from LDS:
    // step kt+1 was requested one iteration ago and goes to the other LDS buffer during this
    // step, step kt+2 is requested now.  Inside a step the operands of 16-deep K slice ks+1 are
    // read from LDS while slice ks is multiplied.
    auto read_ops = [&](const uint16_t* A, const uint16_t* B, int ks, bf16x8 (&a)[TT], bf16x8 (&b)[TW]) {
        const int kc = ks * 16 + (lane >> 5) * 8;
#pragma unroll
        for (int i = 0; i < TT; ++i)
            a[i] = as_bf16x8(*reinterpret_cast<const uint4*>(&A[(wt * TT * 32 + i * 32 + (lane & 31)) * LDS_STRIDE + kc]));
#pragma unroll
        for (int j = 0; j < TW; ++j)
            b[j] = as_bf16x8(*reinterpret_cast<const uint4*>(&B[(ww * TW * 32 + j * 32 + (lane & 31)) * LDS_STRIDE + kc]));
    };
    const GemmViews views = gemm_views(p, PACKED);
    GemmStage<BT, BW, NT> g[2];
    gemm_load<PACKED, EPI>(p, views, t0, n0, 0, true, g[0]);
    gemm_load<PACKED, EPI>(p, views, t0, n0, BK, nk > 1, g[1]);
    gemm_store(g[0], As[0], Bs[0]);
    __syncthreads();
    auto step = [&](int kt, GemmStage<BT, BW, NT>& next, GemmStage<BT, BW, NT>& later) {
        const int buf = kt & 1;
        const uint16_t* A = As[buf];
        const uint16_t* B = Bs[buf];
        bf16x8 a[2][TT], b[2][TW];
        read_ops(A, B, 0, a[0], b[0]);
        gemm_load<PACKED, EPI>(p, views, t0, n0, (kt + 2) * BK, kt + 2 < nk, later);
        // the other buffer was last read before the previous barrier; past the last step the
        // stored stage is zeros that nobody reads, so the store needs no branch
        gemm_store(next, As[buf ^ 1], Bs[buf ^ 1]);
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) {
            if (ks + 1 < BK / 16) read_ops(A, B, ks + 1, a[(ks + 1) & 1], b[(ks + 1) & 1]);
#pragma unroll
            for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int j = 0; j < TW; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[ks & 1][i], b[ks & 1][j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    };
    // both halves of the loop body are unconditional, so each stage keeps its registers
    int kt = 0;
    for (; kt + 1 < nk; kt += 2) {
        step(kt, g[1], g[0]);
        step(kt + 1, g[0], g[1]);
    }
    if (kt < nk) step(kt, g[1], g[0]);

    gemm_epilogue<EPI, TT, TW>(p, acc, t0 + wt * TT * 32, n0, ww, lane);
}

// s_waitcnt on the vector-memory counter only (gfx9 encoding: expcnt and lgkmcnt at maximum).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}
// The same, and every LDS operation of the wave done (lgkmcnt 0).
template <int N>
__device__ __forceinline__ void wait_vmcnt_lds() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0070);
}

// Calls f(std::integral_constant<int, I>) for I = B .. E-1.
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t v, void* lds, uint32_t off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(v, (lds_ptr_t)lds, 16, off, 0, 0, 0);
}

// Plain-weight GEMM whose operand tiles go from memory straight into LDS (buffer loads with
// the LDS destination): no staging registers and no LDS store instructions.  NS LDS stages of
// 64 K values each, NS - 1 stages in flight.  A stage holds BT activation rows then BW weight
// rows of 128 bytes; the 16-byte chunk c of row R sits in slot c ^ ((R >> 1) & 7), which
// spreads both the loads' row segments and the operand reads' 16-row columns over all banks.
// Each wave loads Q 1 KB blocks per stage.  Waves synchronise with a bare s_barrier after
// waiting for their own stage loads and LDS reads, so the later stages stay in flight across
// the barrier.
template <int EPI, int BT, int BW, int WT, int NT, int NS>
__global__ __launch_bounds__(NT) void gemm_dma_kernel(const GemmParams p, int col_tiles, int row_tiles) {
    constexpr int KD = 64, SH = 1;
    constexpr int NW = NT / 64, WW = NW / WT, TT = BT / WT / 32, TW = BW / WW / 32;
    constexpr int ROWB = KD * 2, CPR = ROWB / 16, RPI = 1024 / ROWB;
    constexpr int ROWS = BT + BW, STAGE = ROWS * ROWB, Q = ROWS / RPI / NW;
    static_assert(ROWS % (RPI * NW) == 0 && BT % 16 == 0, "stage blocks per wave");
    static_assert(EPI != GEMM_SWIGLU || TW % 2 == 0, "SwiGLU pairs gate and up tiles inside a wave");
    static_assert(NS == 3 || NS == 4, "two or three stages in flight");
    // one array per stage: the compiler then tells the stages apart and waits for the loads
    // into a stage only before reading that stage (one shared array would make every read
    // wait for every load in flight)
    __shared__ __align__(1024) uint8_t S0[STAGE];
    __shared__ __align__(1024) uint8_t S1[STAGE];
    __shared__ __align__(1024) uint8_t S2[STAGE];
    __shared__ __align__(1024) uint8_t S3[NS > 3 ? STAGE : 16];
    auto stage_of = [&](auto idx) -> uint8_t* {
        constexpr int i = decltype(idx)::value;
        if constexpr (i == 0) return S0;
        else if constexpr (i == 1) return S1;
        else if constexpr (i == 2) return S2;
        else return S3;
    };
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform (scalar)
    const int wt = wave / WW, ww = wave % WW;
    const int tiles = col_tiles * row_tiles;
    const int per = (tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int ct = tile / row_tiles, rt = tile % row_tiles;
    const int t0 = rt * BT;
    const int n0 = ct * (EPI == GEMM_SWIGLU ? BW / 2 : BW);
    const int nk = p.k / KD;
    const uint32_t K = uint32_t(p.k);
    const GemmViews views = gemm_views(p, false);

    // this lane's source offset (K step 0) for each of the wave's Q blocks
    uint32_t goff[Q];
    bool from_x[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int R = (wave * Q + q) * RPI + lane / CPR;
        const uint32_t c = uint32_t((lane % CPR) ^ ((R >> SH) & (CPR - 1)));
        from_x[q] = (wave * Q + q) * RPI < BT;
        const uint32_t row = from_x[q] ? uint32_t(t0 + R) : uint32_t(b_row<EPI>(n0, R - BT));
        goff[q] = (row * K + c * 8) * 2u;
    }
    auto issue = [&](uint8_t* stage, int kt) {
        const uint32_t kill = kt < nk ? 0u : OOB_OFFSET;
        const uint32_t kb = uint32_t(kt) * KD * 2u;
#pragma unroll
        for (int q = 0; q < Q; ++q)
            load_to_lds(from_x[q] ? views.x : views.w, stage + (wave * Q + q) * 1024, (goff[q] + kb) | kill);
    };
    floatx16 acc[TT][TW];
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < TW; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    auto compute = [&](const uint8_t* stage) {
#pragma unroll
        for (int ks = 0; ks < KD / 16; ++ks) {
            const int c = ks * 2 + (lane >> 5);
            bf16x8 a[TT], b[TW];
#pragma unroll
            for (int i = 0; i < TT; ++i) {
                const int R = wt * TT * 32 + i * 32 + (lane & 31);
                a[i] = as_bf16x8(*reinterpret_cast<const uint4*>(stage + R * ROWB + ((c ^ ((R >> SH) & (CPR - 1))) << 4)));
            }
#pragma unroll
            for (int j = 0; j < TW; ++j) {
                const int R = BT + ww * TW * 32 + j * 32 + (lane & 31);
                b[j] = as_bf16x8(*reinterpret_cast<const uint4*>(stage + R * ROWB + ((c ^ ((R >> SH) & (CPR - 1))) << 4)));
            }
#pragma unroll
            for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int j = 0; j < TW; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };
    // step kt: this wave's loads of stage kt are done once at most the loads of the NS - 2
    // later stages are outstanding, and its reads of stage kt - 1 once no LDS operation is
    // (a read issued before the barrier may still be queued in the LDS, and a load into the
    // freed buffer can return before it runs: from L2, or at once when out of range); after
    // the barrier every wave's are, and the buffer of stage kt - 1 is free for stage kt + NS - 1
    auto step = [&](const uint8_t* cur, uint8_t* freed, int kt) {
        __asm__ volatile("" ::: "memory");  // no LDS access of the previous step moves below
        wait_vmcnt_lds<(NS - 2) * Q>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        issue(freed, kt + NS - 1);
        compute(cur);
    };
    static_for<0, NS - 1>([&](auto b) { issue(stage_of(b), decltype(b)::value); });
    int kt = 0;
    for (; kt + NS <= nk; kt += NS)
        static_for<0, NS>([&](auto b) {
            constexpr int i = decltype(b)::value;
            step(stage_of(b), stage_of(std::integral_constant<int, (i + NS - 1) % NS>{}), kt + i);
        });
    static_for<0, NS - 1>([&](auto b) {
        constexpr int i = decltype(b)::value;
        if (kt + i < nk) step(stage_of(b), stage_of(std::integral_constant<int, (i + NS - 1) % NS>{}), kt + i);
    });
    // The last steps issued loads for the stages past the end (out of range: they write zeros
    // into LDS, and keep the per-step load counts uniform).  No wave ends with a load into LDS
    // in flight: the workgroup's LDS may go to the next workgroup on this CU.
    wait_vmcnt<0>();
    gemm_epilogue<EPI, TT, TW>(p, acc, t0 + wt * TT * 32, n0, ww, lane);
}

typedef float floatx4 __attribute__((ext_vector_type(4)));

// A buffer view as its four resource words, and load_to_lds (16 bytes per lane to `lds` + 16 lane)
// as a statement the compiler does not track.  Of loads it tracks, it waits for every one in
// flight before an LDS read that it cannot tell from their destinations, which serialises most
// stage layouts (16 tokens x 6144: 28 us instead of 12); here the kernel's own vmcnt waits order
// loads and reads.  No register is written, so nothing in flight can clobber one.  (s_nop: the
// wait state between a write of M0 and a load into LDS.)
__device__ __forceinline__ u32x4_t view_words(const void* base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return u32x4_t{uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(a)))),
                   uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(a >> 32) & 0xffffu))),
                   uint32_t(__builtin_amdgcn_readfirstlane(int(bytes))), 0x00020000u};
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)p));
}
// M0 is reserved (the compiler keeps no value of its own there across a statement), so naming it
// as clobbered draws a warning at every use; it is named all the same, so that the compiler's own
// writes of M0 stay in order with these.  (As an input operand in M0 the compiler writes it and no
// warning comes, but down of 150 tokens takes 11.2 us instead of 11.0.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_to_lds_untracked(const u32x4_t view, uint32_t lds, uint32_t off, uint32_t scalar_off = 0) {
    __asm__ volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :
                     : "s"(__builtin_amdgcn_readfirstlane(int(lds))), "v"(off), "s"(view),
                       "s"(__builtin_amdgcn_readfirstlane(int(scalar_off)))
                     : "m0", "memory");
}
#pragma clang diagnostic pop

// The same product on tiles of 16x16 blocks, for calls whose tiles of 32-row blocks would leave
// CUs idle: by gemm_tile's rule every call of up to 960 tokens, and longer ones up to 1,536 (o, down;
// 96 x 96) or 1,792 (qkv; 128 x 128).  BT tokens x BM weight rows as 16x16 blocks of
// v_mfma_f32_16x16x32_bf16, whose result equals two v_mfma_f32_32x32x16_bf16 steps bit for bit
// (both fold K in groups of eight in ascending order), at half the latency per K.  A stage is H
// slabs of 64 K values, each [BT activation rows | BM weight rows] of 128 bytes loaded and
// swizzled as in gemm_dma_kernel; NS stages in a ring, NS - 1 in flight.  WT x WM waves own the
// outputs ((BT / WT) x (BM / WM) each); every wave of the workgroup loads.  Weights are the MFMA's
// row operand, so a lane holds four consecutive outputs of one token.
template <int EPI, int BT, int BM, int WT, int WM, int NT, int H, int NS>
__global__ __launch_bounds__(NT) void gemm_small_kernel(const GemmParams p, int col_tiles, int row_tiles, int wide) {
    constexpr int NW = NT / 64, TT = BT / WT / 16, TM = BM / WM / 16;
    constexpr int ROWS = BT + BM, SLAB = ROWS * 128, STAGE = H * SLAB;
    // 1 KB blocks (eight rows) of a stage: XB of activations, WB of weights, dealt to the waves
    // apart, so that no load's source depends on the wave (where the blocks do not divide, the
    // last waves load some twice)
    constexpr int XB = H * BT / 8, WB = H * BM / 8, QX = (XB + NW - 1) / NW, QW = (WB + NW - 1) / NW, Q = QX + QW;
    static_assert(BT % 16 == 0 && BM % 16 == 0 && WT * WM <= NW, "tile");
    static_assert(TT >= 1 && TM >= 1 && TT * WT * 16 == BT && TM * WM * 16 == BM, "wave tile");
    static_assert(EPI != GEMM_SWIGLU || TM % 2 == 0, "SwiGLU pairs gate and up blocks inside a wave");
    static_assert(NS >= 2 && (NS - 2) * Q < 64, "loads in flight");
    __shared__ __align__(1024) uint8_t S[NS * STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles = col_tiles * row_tiles;
    const int per = (tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int ct = tile / row_tiles, rt = tile % row_tiles;
    const int t0 = rt * BT;
    const int n0 = ct * (EPI == GEMM_SWIGLU ? BM / 2 : BM);
    const uint32_t K = uint32_t(p.k);
    const int nk = p.k / (64 * H);
    const u32x4_t xv = view_words(p.x, uint32_t(p.tokens) * K * 2u), wv = view_words(p.w, uint32_t(p.m) * K * 2u);
    const uint32_t lds = lds_address(S);

    // this lane's source offset (stage 0) for each of the wave's blocks
    uint32_t xoff[QX], woff[QW], xdst[QX], wdst[QW];
#pragma unroll
    for (int q = 0; q < QX; ++q) {
        const int id = (wave * QX + q) % XB, h = id / (BT / 8), R = id % (BT / 8) * 8 + (lane >> 3);
        const uint32_t c = uint32_t((lane & 7) ^ ((R >> 1) & 7));
        xoff[q] = (uint32_t(t0 + R) * K + uint32_t(h) * 64u + c * 8) * 2u;
        xdst[q] = uint32_t(h * SLAB + id % (BT / 8) * 1024);
    }
#pragma unroll
    for (int q = 0; q < QW; ++q) {
        const int id = (wave * QW + q) % WB, h = id / (BM / 8), r = id % (BM / 8) * 8 + (lane >> 3);
        const uint32_t c = uint32_t((lane & 7) ^ (((BT + r) >> 1) & 7));
        uint32_t row;
        if constexpr (EPI == GEMM_SWIGLU)  // 16 gate rows, then their 16 up rows
            row = uint32_t(((r >> 4) & 1 ? INTER : 0) + n0 + (r >> 5) * 16 + (r & 15));
        else row = uint32_t(n0 + r);
        woff[q] = (row * K + uint32_t(h) * 64u + c * 8) * 2u;
        wdst[q] = uint32_t(h * SLAB + BT * 128 + id % (BM / 8) * 1024);
    }
    auto issue = [&](uint32_t stage, int kt) {  // stage: its byte offset in S
        const uint32_t kill = kt < nk ? 0u : OOB_OFFSET;
        const uint32_t kb = uint32_t(kt) * (H * 128u);
#pragma unroll
        for (int q = 0; q < QX; ++q) load_to_lds_untracked(xv, lds + stage + xdst[q], (xoff[q] + kb) | kill);
#pragma unroll
        for (int q = 0; q < QW; ++q) load_to_lds_untracked(wv, lds + stage + wdst[q], (woff[q] + kb) | kill);
    };
    const bool computes = WT * WM == NW || wave < WT * WM;
    const int wt = wave / WM, wm = wave % WM;
    floatx4 acc[TM][TT];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const uint8_t* stage) {
#pragma unroll
        for (int s = 0; s < 2 * H; ++s) {
            const uint8_t* slab = stage + (s >> 1) * SLAB;
            const int c = (s & 1) * 4 + (lane >> 4), r = lane & 15;
            bf16x8 a[TM], b[TT];
#pragma unroll
            for (int j = 0; j < TT; ++j) {
                const int R = (wt * TT + j) * 16 + r;
                b[j] = as_bf16x8(*reinterpret_cast<const uint4*>(slab + R * 128 + ((c ^ ((R >> 1) & 7)) << 4)));
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int R = BT + (wm * TM + i) * 16 + r;
                a[i] = as_bf16x8(*reinterpret_cast<const uint4*>(slab + R * 128 + ((c ^ ((R >> 1) & 7)) << 4)));
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TT; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };
    // the waits of gemm_dma_kernel: own loads of this stage and own LDS reads of the last done,
    // then the barrier; the stage before is then free
    for (int b = 0; b < NS - 1; ++b) issue(uint32_t(b) * STAGE, b);
    uint32_t cur = 0, freed = (NS - 1) * STAGE;
    for (int kt = 0; kt < nk; ++kt) {
        __asm__ volatile("" ::: "memory");
        wait_vmcnt_lds<(NS - 2) * Q>();
        __builtin_amdgcn_s_barrier();
        __asm__ volatile("" ::: "memory");
        issue(freed, kt + NS - 1);
        if (computes) compute(S + cur);
        freed = cur;
        cur = cur + STAGE == NS * STAGE ? 0u : cur + STAGE;
    }
    wait_vmcnt<0>();  // no wave ends with a load into LDS in flight
    if (!computes) return;

    // Element r of a block is weight row 4 (lane / 16) + r, token lane % 16.  `wide`: the four
    // outputs of a lane are stored together (m a multiple of four, y aligned to four outputs).
    const uint32_t M = uint32_t(p.m);
    const uint32_t cols = EPI == GEMM_SWIGLU ? uint32_t(INTER) : M;
    constexpr uint32_t ES = EPI == GEMM_SWIGLU || EPI == GEMM_BF16 ? 2u : 4u;
    const __amdgpu_buffer_rsrc_t yv =
        buffer_view(ES == 2u ? static_cast<const void*>(p.y16) : static_cast<const void*>(p.y), uint32_t(p.tokens) * cols * ES);
#pragma unroll
    for (int j = 0; j < TT; ++j) {
        const uint32_t t = uint32_t(t0 + (wt * TT + j) * 16 + (lane & 15));
#pragma unroll
        for (int i = 0; i < TM; i += EPI == GEMM_SWIGLU ? 2 : 1) {
            const uint32_t m = uint32_t(n0 + (EPI == GEMM_SWIGLU ? (wm * TM + i) >> 1 : wm * TM + i) * 16 + (lane >> 4) * 4);
            uint32_t w[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if constexpr (EPI == GEMM_SWIGLU) {  // as gemm_epilogue
                    const float gt = roundbf(acc[i][j][r]);
                    const float up = roundbf(acc[i + 1][j][r]);
                    const float silu = gt / (1.0f + exp_det(-gt));
                    w[r] = bits(roundbf(silu) * up);
                } else if constexpr (EPI == GEMM_BF16) {
                    w[r] = bits(acc[i][j][r]);
                } else if constexpr (EPI == GEMM_F32) {
                    w[r] = __float_as_uint(roundbf(acc[i][j][r]));
                } else {
                    w[r] = __float_as_uint(acc[i][j][r]);
                }
            }
            const uint32_t e = t * cols + m;
            if (wide) {
                const uint32_t off = m < cols ? e * ES : OOB_OFFSET;
                if constexpr (ES == 2u) {
                    const u32x2_t v = {(w[0] & 0xffffu) | (w[1] << 16), (w[2] & 0xffffu) | (w[3] << 16)};
                    __builtin_amdgcn_raw_buffer_store_b64(v, yv, off, 0, 0);
                } else {
                    const u32x4_t v = {w[0], w[1], w[2], w[3]};
                    __builtin_amdgcn_raw_buffer_store_b128(v, yv, off, 0, 0);
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t off = m + uint32_t(r) < cols ? (e + uint32_t(r)) * ES : OOB_OFFSET;
                    if constexpr (ES == 2u) buffer_store2(yv, off, uint16_t(w[r]));
                    else buffer_store4(yv, off, w[r]);
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------ norms
// Post-norm + residual + next norm of prefill rows (Kernels.metal:46-90).  One wave per
// token, four tokens per workgroup: lane l owns elements 512c + 8l .. +8 (c < 3), read and
// written as 16-byte rows; both sums of squares are wave reductions.
__global__ __launch_bounds__(256) void rows_norm_kernel(const RowsNormParams p) {
    constexpr int C = HIDDEN / 512;
    const int lane = threadIdx.x & 63;
    const int t = int(blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    if (t >= p.tokens) return;
    auto unpack = [](const uint4 w, float (&f)[8]) {
        const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) { f[2 * k] = lo(u[k]); f[2 * k + 1] = hi(u[k]); }
    };
    float xv[C][8];
    const size_t row = size_t(t) * HIDDEN;
    // the next norm's gains are requested with the row's inputs (off the reductions' path)
    uint4 gnw[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        gnw[c] = p.xn ? *reinterpret_cast<const uint4*>(p.g_next + 512 * c + 8 * lane) : make_uint4(0, 0, 0, 0);
    if (p.tokens_in) {
        int tok = p.tokens_in[t];
        tok = (tok < 0 || tok >= VOCAB) ? 0 : tok;
#pragma unroll
        for (int c = 0; c < C; ++c)
            unpack(*reinterpret_cast<const uint4*>(p.embed + size_t(tok) * HIDDEN + 512 * c + 8 * lane), xv[c]);
    } else {
        float pv[C][8], rv[C][8], gp[C][8];
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int i = 512 * c + 8 * lane;
            unpack(*reinterpret_cast<const uint4*>(p.in + row + i), pv[c]);
            unpack(*reinterpret_cast<const uint4*>(p.x + row + i), rv[c]);
            unpack(*reinterpret_cast<const uint4*>(p.g_post + i), gp[c]);
        }
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < 8; ++k) ss += pv[c][k] * pv[c][k];
        const float r = 1.0f / sqrtf(wave_sum(ss) / float(HIDDEN) + 1e-6f);
        // z = roundbf(roundbf(p r) roundbf(w + offset)), x = roundbf(x + z): the roundings two
        // at a time with the packed RNE conversion (same bits as `roundbf`)
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < 8; k += 2) {
                float t0, t1, g0, g1, z0, z1;
                round_bf16x2(pv[c][k] * r, pv[c][k + 1] * r, t0, t1);
                round_bf16x2(gp[c][k] + p.post_offset, gp[c][k + 1] + p.post_offset, g0, g1);
                round_bf16x2(t0 * g0, t1 * g1, z0, z1);
                round_bf16x2(rv[c][k] + z0, rv[c][k + 1] + z1, xv[c][k], xv[c][k + 1]);
            }
    }
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < 8; ++k) ss += xv[c][k] * xv[c][k];
    const float r = 1.0f / sqrtf(wave_sum(ss) / float(HIDDEN) + 1e-6f);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int i = 512 * c + 8 * lane;
        uint32_t xw[4], nw[4];
        float gn[8];
        unpack(gnw[c], gn);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            xw[k] = pack_bf16(xv[c][2 * k], xv[c][2 * k + 1]);  // BF16 values: exact
            if (p.xn) {
                float t0, t1, g0, g1;
                round_bf16x2(xv[c][2 * k] * r, xv[c][2 * k + 1] * r, t0, t1);
                round_bf16x2(gn[2 * k] + 1.0f, gn[2 * k + 1] + 1.0f, g0, g1);
                nw[k] = pack_bf16(t0 * g0, t1 * g1);
            }
        }
        *reinterpret_cast<uint4*>(p.x + row + i) = make_uint4(xw[0], xw[1], xw[2], xw[3]);
        if (p.xn) *reinterpret_cast<uint4*>(p.xn + row + i) = make_uint4(nw[0], nw[1], nw[2], nw[3]);
    }
}

// ---------------------------------------------------------------------------- qk prep
// One workgroup per token (the `qkv` kernel, Kernels.metal:223-259, for a prefill chunk):
// thread (h, s) = (tid/16, tid%16) normalises and rotates RoPE pairs (d, d+64) for
// d = 4s..4s+3 of query head h -- global layers at the absolute position, local layers at
// pos - base with base = max(0, chunk_start - 2047) of the token's 16-token chunk
// (Runtime.swift:389, Kernels.metal:251,283-284).  Threads 0..15 do the same for the key
// (rotated only on global layers; local keys are cached unrotated) and write it to slot
// pos % capacity; threads 64..191 copy the value row.
__global__ __launch_bounds__(256) void qk_prep_kernel(const QkPrepParams p) {
    const int t = blockIdx.x, tid = threadIdx.x;
    const int hq = tid >> 4, sq = tid & 15;
    uint32_t ts = uint32_t(t);  // the token within its segment
    uint16_t *keys = p.keys, *values = p.values, *keys_rot = p.keys_rot;
    if (p.seg.n > 1) {
        const PrefillSegment sg = p.seg.of_token(t);
        ts -= uint32_t(sg.token0);
        keys += size_t(sg.lane) * p.capacity * HEAD_DIM;
        values += size_t(sg.lane) * p.capacity * HEAD_DIM;
        if (keys_rot) keys_rot += size_t(sg.lane) * p.rot_rows * HEAD_DIM;
    }
    const uint32_t pos = p.p0 + ts;
    const uint32_t chunk = p.p0 + (ts / CHUNK) * CHUNK;
    const uint32_t base = chunk > uint32_t(WINDOW - 1) ? chunk - uint32_t(WINDOW - 1) : 0u;
    const uint32_t qcoord = p.full ? pos : pos - base;
    const uint16_t* x = p.qkv + size_t(t) * QKV;
    // four BF16 values as FP32
    auto load4 = [](const uint16_t* s) {
        const uint2 w = *reinterpret_cast<const uint2*>(s);
        return make_float4(lo(w.x), hi(w.x), lo(w.y), hi(w.y));
    };
    // the key part's inputs (threads 0..15) are requested with the queries'
    const bool kthread = tid < 16;
    const bool krot = !p.full && keys_rot && pos < p.rot_rows;
    float4 klo = make_float4(0.f, 0.f, 0.f, 0.f), khi = klo;
    uint2 kgl = make_uint2(0, 0), kgh = kgl;
    uint4 kr4 = make_uint4(0, 0, 0, 0);
    if (kthread) {
        klo = load4(x + ATTN + tid * 4);
        khi = load4(x + ATTN + 64 + tid * 4);
        kgl = *reinterpret_cast<const uint2*>(p.k_norm + tid * 4);
        kgh = *reinterpret_cast<const uint2*>(p.k_norm + 64 + tid * 4);
        if (p.full || krot)
            kr4 = *reinterpret_cast<const uint4*>((p.full ? p.global_rope : p.local_rope) + size_t(pos) * 64 + tid * 4);
    }
    {
        const float4 qlo = load4(x + hq * HEAD_DIM + sq * 4);
        const float4 qhi = load4(x + hq * HEAD_DIM + 64 + sq * 4);
        const uint2 glo = *reinterpret_cast<const uint2*>(p.q_norm + sq * 4);
        const uint2 ghi = *reinterpret_cast<const uint2*>(p.q_norm + 64 + sq * 4);
        const uint4 qr = *reinterpret_cast<const uint4*>((p.full ? p.global_rope : p.local_rope) + size_t(qcoord) * 64 + sq * 4);
        float z[8];
        head_norm8(qlo, qhi, glo, ghi, z);
        const uint32_t c4[4] = {qr.x, qr.y, qr.z, qr.w};
        // rope_pair_x2f: two RoPE pairs per packed RNE conversion (same bits as rope_pair)
#pragma unroll
        for (int j = 0; j < 4; j += 2) rope_pair_x2f(z[j], z[4 + j], c4[j], z[j + 1], z[4 + j + 1], c4[j + 1]);
        uint16_t* qo = p.q16 + (size_t(t) * HEADS + hq) * HEAD_DIM;
        *reinterpret_cast<uint2*>(qo + sq * 4) = make_uint2(pack_bf16(z[0], z[1]), pack_bf16(z[2], z[3]));
        *reinterpret_cast<uint2*>(qo + 64 + sq * 4) = make_uint2(pack_bf16(z[4], z[5]), pack_bf16(z[6], z[7]));
    }
    const size_t slot = size_t(pos % p.capacity) * HEAD_DIM;
    if (kthread) {
        float z[8];
        head_norm8(klo, khi, kgl, kgh, z);
        const uint32_t c4[4] = {kr4.x, kr4.y, kr4.z, kr4.w};
        if (p.full) {
#pragma unroll
            for (int j = 0; j < 4; j += 2) rope_pair_x2f(z[j], z[4 + j], c4[j], z[j + 1], z[4 + j + 1], c4[j + 1]);
        } else if (krot) {
            // the copy rotated at the key's own position (decode inside the first window)
            float zr[8] = {z[0], z[1], z[2], z[3], z[4], z[5], z[6], z[7]};
#pragma unroll
            for (int j = 0; j < 4; j += 2) rope_pair_x2f(zr[j], zr[4 + j], c4[j], zr[j + 1], zr[4 + j + 1], c4[j + 1]);
            uint16_t* kr = keys_rot + size_t(pos) * HEAD_DIM;
            *reinterpret_cast<uint2*>(kr + tid * 4) = make_uint2(pack_bf16(zr[0], zr[1]), pack_bf16(zr[2], zr[3]));
            *reinterpret_cast<uint2*>(kr + 64 + tid * 4) = make_uint2(pack_bf16(zr[4], zr[5]), pack_bf16(zr[6], zr[7]));
        }
        auto word = [](float a, float b) { return (bits(a) & 0xffffu) | (bits(b) << 16); };
        *reinterpret_cast<uint2*>(keys + slot + tid * 4) = make_uint2(word(z[0], z[1]), word(z[2], z[3]));
        *reinterpret_cast<uint2*>(keys + slot + 64 + tid * 4) = make_uint2(word(z[4], z[5]), word(z[6], z[7]));
    }
    if (tid >= 64 && tid < 64 + HEAD_DIM) {
        const int d = tid - 64;
        values[slot + d] = x[ATTN + HEAD_DIM + d];
    }
}

__global__ __launch_bounds__(HIDDEN / 8) void gather_last_kernel(const uint16_t* a, const uint16_t* b,
                                                                const PrefillSegments seg, uint16_t* a_out, uint16_t* b_out) {
    const PrefillSegment sg = seg.s[blockIdx.x];
    const size_t from = size_t(sg.token0 + sg.tokens - 1) * HIDDEN + threadIdx.x * 8, to = size_t(blockIdx.x) * HIDDEN + threadIdx.x * 8;
    *reinterpret_cast<uint4*>(a_out + to) = *reinterpret_cast<const uint4*>(a + from);
    *reinterpret_cast<uint4*>(b_out + to) = *reinterpret_cast<const uint4*>(b + from);
}

// --------------------------------------------------------------------- flash attention
// Prefill attention (Runtime.swift:389-444: scores, scale 1/sqrt(128) before the max,
// softmax, roundbf(sum p v)) as MFMA flash attention over the cached keys.
//
// A workgroup takes 8 tokens x 16 heads = 128 query columns; wave w owns tokens 2w, 2w+1:
// lane column c = lane%32 is token 2w + c/16, head c%16 (MQA: every head reads the same
// keys, so one K/V tile serves all 128 columns).  With keys as rows,
//   S^T = K Q^T   and   O^T = V^T P^T,
// a query's 64 scores of a tile sit in one lane column (two halves of 32 lanes), so the
// online-softmax statistics need a single cross-half exchange, and the S^T accumulator is
// already the B operand layout of the P.V product.  P is split as hi + lo BF16 so the
// P.V product keeps ~16 significant bits of the FP32 probabilities.  The softmax weights come
// from `exp2_det` and nothing is contracted, so every output is a fixed function of the
// inputs that a CPU restatement reproduces bit for bit.
//
// Two kernels share that arithmetic: the staged one (K/V tiles through registers into K rows
// and V^T in LDS; the only one that can rotate keys while staging) and the direct one (K/V
// tiles loaded straight into LDS, V^T operands by transposing LDS reads), used when no block
// of a call rotates its keys: global layers, and local layers inside the rotated-key cache.
//
// Keys of local layers are rotated while staged, with coordinate key_pos - base of the
// workgroup's 16-token chunk (base = max(0, chunk_start - 2047)); where base is 0 and every
// key of the block lies in the rotated-key cache, that coordinate is the key's position and
// the cached rotations (written by qk_prep_kernel) are staged as they are.
constexpr int FT = 8;                 // tokens per query block (workgroup)
constexpr int FK = 64;                // keys per tile
static_assert(FT == 8 && FK == 64, "flash_block_tiles (prefill.h) assumes these sizes");
constexpr int KST = HEAD_DIM + 8;     // K tile row stride (BF16), 16-byte aligned rows
constexpr int VST = FK + 4;           // V^T tile row stride (BF16): 34 dwords, so 16 lanes reading
                                      // 8 bytes from 16 consecutive rows hit 32 distinct banks
constexpr float SCALE_LOG2E = 0.08838834764831845f * 1.4426950408889634f;

struct KvStage {
    uint4 ka[2], kb[2], rr[4], v[4];
};
// Where a tile's keys come from: unrotated (rotate while staged), rotated (global layers, or
// the rotated-key cache of a local layer).
struct KvSource {
    const uint16_t* keys;
    bool rotate;
};

// Global loads of one tile: thread -> key tid/4 with RoPE pairs (d, d+64), d = 16*(tid%4)
// .. +16; and values of keys 4*(tid%16) .. +4 at dims 8*(tid/16) .. +8.  Keys past khi (the
// last tile's tail) load key khi instead: their scores are masked and their weights are
// exactly 0, so any finite row serves, every load stays on a written key, and no register
// has to be cleared or load predicated.
__device__ __forceinline__ void flash_load(const FlashParams& p, const KvSource& src, uint32_t k0, uint32_t khi,
                                           uint32_t base, KvStage& s) {
    const int tid = threadIdx.x;
    const int part = tid & 3;
    // ring slots: one modulo per tile, then at most one wrap per key when the ring holds a
    // whole tile (offsets are below 64); smaller rings wrap by repeated subtraction
    const uint32_t slot0 = k0 % p.capacity;
    const bool big_ring = p.capacity >= uint32_t(FK);
    auto ring = [&](uint32_t off) {
        uint32_t slot = slot0 + off;
        if (big_ring) return slot >= p.capacity ? slot - p.capacity : slot;
        while (slot >= p.capacity) slot -= p.capacity;
        return slot;
    };
    const uint32_t kp = min(k0 + uint32_t(tid >> 2), khi);
    // the rotated-key cache is indexed by position (kp < rot_rows), the ring by slot
    const uint16_t* row = src.keys + size_t(src.rotate || p.full ? ring(kp - k0) : kp) * HEAD_DIM;
    s.ka[0] = *reinterpret_cast<const uint4*>(row + part * 16);
    s.ka[1] = *reinterpret_cast<const uint4*>(row + part * 16 + 8);
    s.kb[0] = *reinterpret_cast<const uint4*>(row + 64 + part * 16);
    s.kb[1] = *reinterpret_cast<const uint4*>(row + 64 + part * 16 + 8);
    if (src.rotate) {
        const uint4* rr = reinterpret_cast<const uint4*>(p.local_rope + size_t(kp - base) * 64 + part * 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) s.rr[i] = rr[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t kv = min(k0 + uint32_t(4 * (tid & 15) + i), khi);
        s.v[i] = *reinterpret_cast<const uint4*>(p.values + size_t(ring(kv - k0)) * HEAD_DIM + 8 * (tid >> 4));
    }
}

__device__ __forceinline__ uint32_t u16_of(const uint4& v, int k) {
    const uint32_t w = k < 2 ? v.x : k < 4 ? v.y : k < 6 ? v.z : v.w;
    return (k & 1) ? (w >> 16) : (w & 0xffffu);
}

__device__ __forceinline__ void flash_store(const KvSource& src, const KvStage& s, uint16_t* Ks, uint16_t* Vt) {
    const int tid = threadIdx.x;
    const int part = tid & 3, key = tid >> 2;
    uint16_t* krow = Ks + key * KST;
    if (!src.rotate) {
        *reinterpret_cast<uint4*>(krow + part * 16) = s.ka[0];
        *reinterpret_cast<uint4*>(krow + part * 16 + 8) = s.ka[1];
        *reinterpret_cast<uint4*>(krow + 64 + part * 16) = s.kb[0];
        *reinterpret_cast<uint4*>(krow + 64 + part * 16 + 8) = s.kb[1];
    } else {
        const uint32_t aw[8] = {s.ka[0].x, s.ka[0].y, s.ka[0].z, s.ka[0].w, s.ka[1].x, s.ka[1].y, s.ka[1].z, s.ka[1].w};
        const uint32_t bw[8] = {s.kb[0].x, s.kb[0].y, s.kb[0].z, s.kb[0].w, s.kb[1].x, s.kb[1].y, s.kb[1].z, s.kb[1].w};
        const uint32_t rw[16] = {s.rr[0].x, s.rr[0].y, s.rr[0].z, s.rr[0].w, s.rr[1].x, s.rr[1].y, s.rr[1].z, s.rr[1].w,
                                 s.rr[2].x, s.rr[2].y, s.rr[2].z, s.rr[2].w, s.rr[3].x, s.rr[3].y, s.rr[3].z, s.rr[3].w};
        uint32_t ao[8], bo[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) rope_pair_x2(aw[i], bw[i], rw[2 * i], rw[2 * i + 1], ao[i], bo[i]);
        *reinterpret_cast<uint4*>(krow + part * 16) = make_uint4(ao[0], ao[1], ao[2], ao[3]);
        *reinterpret_cast<uint4*>(krow + part * 16 + 8) = make_uint4(ao[4], ao[5], ao[6], ao[7]);
        *reinterpret_cast<uint4*>(krow + 64 + part * 16) = make_uint4(bo[0], bo[1], bo[2], bo[3]);
        *reinterpret_cast<uint4*>(krow + 64 + part * 16 + 8) = make_uint4(bo[4], bo[5], bo[6], bo[7]);
    }
    // V^T: 4 keys of one dim per 8-byte store
    const int kg = 4 * (tid & 15), d0 = 8 * (tid >> 4);  // consecutive lanes: consecutive key groups
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t w0 = u16_of(s.v[0], j) | (u16_of(s.v[1], j) << 16);
        const uint32_t w1 = u16_of(s.v[2], j) | (u16_of(s.v[3], j) << 16);
        *reinterpret_cast<uint2*>(Vt + (d0 + j) * VST + kg) = make_uint2(w0, w1);
    }
}

// Two FP32 values in [0, 1] as BF16 pairs hi + lo (RNE, v_cvt_pk_bf16_f32): hi + lo carries ~16
// significant bits of each value.
__device__ __forceinline__ void split_bf16(float a, float b, uint32_t& hw, uint32_t& lw) {
    hw = pack_bf16(a, b);
    lw = pack_bf16(a - lo(hw), b - hi(hw));
}
// The same split for the direct kernel, whose vector instructions run beside its products: the
// differences value - hi are exact, so one v_dot2_f32_bf16 each (hi times -1 and 0 onto the value)
// gives the same bits in fewer instructions.  (The factors stay in registers: as literals the
// compiler encodes one as the inline constant -1.0, which this instruction does not read as the
// pair (0, -1).)  In the staged kernel, which waits for each result, it is the slower one: 500
// local queries from position 0 32.0 us instead of 30.8.
__device__ __forceinline__ void split_bf16_dot2(float a, float b, uint32_t& hw, uint32_t& lw) {
    uint32_t first = 0x0000bf80u, second = 0xbf800000u;
    __asm__("" : "+s"(first), "+s"(second));
    hw = pack_bf16(a, b);
    lw = pack_bf16(dot2bf(hw, first, a), dot2bf(hw, second, b));
}

// Part `part` of query block qb.  QSA: global layers with a selection bitmap (a separate
// instance, so the dense kernel's edge tiles carry no bitmap test).  SHORT: no block of the call
// has more than two tiles, and the last requests and scores nothing ahead.  In the longer calls'
// kernel a stale copy is requested, waited for and scored there: 3 global queries take 8.3 us in it
// and 7.0 in this one, 100 10.1 and 9.2.  (Both in one kernel cost its loop up to 260 bytes of
// spilled registers and 500 queries up to 29 us instead of 23.)
template <bool QSA, bool DIRECT, bool SHORT>
__device__ __forceinline__ void flash_prefill(const FlashParams& pass, const int block, const int part) {
#pragma clang fp contract(off)  // fixed rounding sequence, reproduced by the CPU oracle
    // block `block` of the pass is block qb of its segment
    PrefillSegment sg = pass.seg.s[0];
    FlashParams p = pass;
    if (pass.seg.n > 1) {
        sg = pass.seg.of_block(block);
        p.q += size_t(sg.token0) * ATTN;
        p.out += size_t(sg.token0) * ATTN;
        p.keys += size_t(sg.lane) * p.capacity * HEAD_DIM;
        p.values += size_t(sg.lane) * p.capacity * HEAD_DIM;
        if (p.keys_rot) p.keys_rot += size_t(sg.lane) * p.rot_rows * HEAD_DIM;
    }
    const int qb = block - sg.first_block, tokens = sg.tokens;
    // two key and two value tiles: 16 KB each on the direct path (L); padded K rows and V^T on the
    // staged one, four arrays that the compiler tells apart (L0 .. L3; parts of one array: 333
    // local queries from position 3001 45.7 us instead of 45.1)
    constexpr int KT = FK * KST, VT = HEAD_DIM * VST;
    __shared__ __align__(1024) uint8_t L[DIRECT ? 4 * FK * HEAD_DIM * 2 : 16];
    __shared__ __align__(1024) uint16_t L0[DIRECT ? 8 : KT];
    __shared__ __align__(1024) uint16_t L1[DIRECT ? 8 : KT];
    __shared__ __align__(1024) uint16_t L2[DIRECT ? 8 : VT];
    __shared__ __align__(1024) uint16_t L3[DIRECT ? 8 : VT];
    __shared__ int s_last;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, half = lane >> 5;
    const int t0 = qb * FT;
    const int t1 = min(t0 + FT, tokens);
    const int tq = t0 + wave * 2 + (col >> 4);
    const int head = col & 15;
    const bool qvalid = tq < tokens;
    const int tqc = qvalid ? tq : t1 - 1;
    const uint32_t qpos = p.p0 + uint32_t(tqc);
    const uint32_t chunk = p.p0 + (uint32_t(t0) / CHUNK) * CHUNK;
    const uint32_t base = p.full ? 0u : (chunk > uint32_t(WINDOW - 1) ? chunk - uint32_t(WINDOW - 1) : 0u);
    const uint32_t plo = p.p0 + uint32_t(t0), khi = p.p0 + uint32_t(t1 - 1);
    const uint32_t klo = p.full ? 0u : (plo > uint32_t(WINDOW - 1) ? plo - uint32_t(WINDOW - 1) : 0u);
    // The block's key tiles are split over up to FLASH_PARTS workgroups of about
    // FLASH_PART_TILES tiles each, so long (late) query blocks do not set the kernel's length.
    const int ntiles = flash_block_tiles(tokens, p.p0, p.full, qb);
    const int parts = flash_block_parts(ntiles);
    if (part >= parts) return;
    const int j0 = part * ntiles / parts, j1 = (part + 1) * ntiles / parts;

    // Q^T fragments (B operand of S^T): k-step s covers dims 16s + 8*half .. +8
    bf16x8 qf[8];
    {
        const uint16_t* qrow = p.q + (size_t(tqc) * HEADS + head) * HEAD_DIM;
#pragma unroll
        for (int s = 0; s < 8; ++s) qf[s] = as_bf16x8(*reinterpret_cast<const uint4*>(qrow + 16 * s + 8 * half));
    }
    floatx16 oacc[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.f;
    float m = NEG_INF, ls = 0.f;

    // QSA: the query's blocks of four keys complete at its position are seen only when
    // selected (bit b of its bitmap word b / 32); its unfinished block always is
    const uint32_t* qmask = QSA ? p.qsa_mask + size_t(tqc) * p.qsa_words : nullptr;
    const uint32_t qcomplete = (qpos + 1) / 4;
    const bool cached = !p.full && p.keys_rot != nullptr && base == 0 && khi < p.rot_rows;
    const KvSource src{cached ? p.keys_rot : p.keys, !p.full && !cached};

    // Online softmax of tile j in the base-2 domain: x = score * scale * log2(e),
    // p = 2^(x - max).  Element i of tile r is key k0 + 32r + 8(i/4) + 4*half + i%4.  Only
    // tiles that cross a query's causal edge or window start need the mask.  QSA: every tile
    // is masked by the query's selected blocks (its unfinished block is always seen).  Leaves
    // the probabilities in sacc and rescales oacc.
    auto softmax = [&](int j, floatx16 (&sacc)[2]) {
        const uint32_t k0 = klo + uint32_t(j * FK);
        const bool edge = QSA || !(k0 + uint32_t(FK - 1) <= plo && (p.full || k0 + uint32_t(WINDOW - 1) >= khi));
        float mt = NEG_INF;
        if (edge) {
            // QSA (global layers: k0 is a multiple of 64): the tile's 16 blocks b0 .. b0 + 15
            // are bits 0..15 of one bitmap word shifted by b0 % 32, read once per tile; blocks
            // at or past qcomplete are not tested
            uint32_t qbits = 0u;
            const uint32_t b0 = k0 >> 2;
            if (QSA && b0 < qcomplete) qbits = qmask[b0 >> 5] >> (b0 & 31);
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const uint32_t kp = k0 + uint32_t(32 * r + 8 * (i >> 2) + 4 * half + (i & 3));
                    bool vis = kp <= qpos && (p.full || kp + uint32_t(WINDOW - 1) >= qpos);
                    if (QSA) {
                        const uint32_t b = kp >> 2;
                        vis = vis && (b >= qcomplete || ((qbits >> (b - b0)) & 1u));
                    }
                    const float x = vis ? sacc[r][i] * SCALE_LOG2E : NEG_INF;
                    sacc[r][i] = x;
                    mt = fmaxf(mt, x);
                }
        } else {
#pragma unroll
            for (int r = 0; r < 2; ++r)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float x = sacc[r][i] * SCALE_LOG2E;
                    sacc[r][i] = x;
                    mt = fmaxf(mt, x);
                }
        }
        mt = fmaxf(mt, xor_lane<32>(mt));
        const float mn = fmaxf(m, mt);
        const float ms = mn == NEG_INF ? 0.0f : mn;  // nothing visible yet: every p is 0
        const float alpha = exp2_det(m - ms);
        ls *= alpha;
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float e = exp2_det(sacc[r][i] - ms);
                sacc[r][i] = e;
                ls += e;
            }
        m = mn;
        // alpha is exactly 1 where the running maximum did not move: the wave skips the
        // rescale when that holds in every lane (multiplying by 1 changes nothing)
        if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                for (int i = 0; i < 16; ++i) oacc[dt][i] *= alpha;
        }
    };
    // O^T += V^T P^T; k-step s takes keys 16s + 4*half + {0..3} and 16s + 8 + 4*half + {0..3};
    // vt(dt, s) returns the V^T operand of d-tile dt at k-step s
    auto pv = [&](const floatx16 (&sacc)[2], auto vt) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int r = s >> 1, i0 = (s & 1) * 8;
            uint32_t hw[4], lw[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) split_bf16(sacc[r][i0 + 2 * k], sacc[r][i0 + 2 * k + 1], hw[k], lw[k]);
            const bf16x8 ph = as_bf16x8(make_uint4(hw[0], hw[1], hw[2], hw[3]));
            const bf16x8 pl = as_bf16x8(make_uint4(lw[0], lw[1], lw[2], lw[3]));
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                const bf16x8 a = vt(dt, s);
                oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, ph, oacc[dt], 0, 0, 0);
                oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pl, oacc[dt], 0, 0, 0);
            }
        }
    };
    // S^T = K Q^T for 64 keys (two 32-row tiles); kop(r, s) returns the K operand of row tile
    // r at k-step s
    auto qk = [&](floatx16 (&sacc)[2], auto kop) {
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int i = 0; i < 16; ++i) sacc[r][i] = 0.f;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
#pragma unroll
            for (int r = 0; r < 2; ++r) sacc[r] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kop(r, s), qf[s], sacc[r], 0, 0, 0);
        }
    };

    if constexpr (!DIRECT) {
        // staged through registers (keys rotated on the way where the block needs it): K rows
        // and V^T in LDS
        KvStage st;
        flash_load(p, src, klo + uint32_t(j0 * FK), khi, base, st);
        flash_store(src, st, L0, L2);
        __syncthreads();
        for (int j = j0; j < j1; ++j) {
            const bool odd = ((j - j0) & 1) != 0;
            const uint16_t* Kc = odd ? L1 : L0;
            const uint16_t* Vc = odd ? L3 : L2;
            if (j + 1 < j1) flash_load(p, src, klo + uint32_t((j + 1) * FK), khi, base, st);
            floatx16 sacc[2];
            qk(sacc, [&](int r, int s) {
                return as_bf16x8(*reinterpret_cast<const uint4*>(&Kc[(r * 32 + col) * KST + 16 * s + 8 * half]));
            });
            softmax(j, sacc);
            pv(sacc, [&](int dt, int s) {
                const uint16_t* vrow = &Vc[(dt * 32 + col) * VST + 16 * s + 4 * half];
                const uint2 x0 = *reinterpret_cast<const uint2*>(vrow);
                const uint2 x1 = *reinterpret_cast<const uint2*>(vrow + 8);
                return as_bf16x8(make_uint4(x0.x, x0.y, x1.x, x1.y));
            });
            if (j + 1 < j1) flash_store(src, st, odd ? L0 : L1, odd ? L2 : L3);
            __syncthreads();
        }
    } else {
        // (DIRECT: the launch holds only blocks whose keys need no rotation)
        // Keys (already rotated) and values loaded straight into LDS, two 16 KB tiles of each
        // (tile j in buffer (j - j0) % 2).  Rows are 256 bytes, swizzled so that both operand
        // reads hit every bank: 16-byte chunk c of key row R in slot c ^ (R % 16), 64-byte
        // chunk d of value row R in slot d ^ (R % 4).  Tile j runs S^T of tile j + 1 beside the
        // scaling and maximum of its own scores, then each quarter's exponentials beside the
        // P.V products of the quarter before, in an order fixed by scheduling fences: a wave
        // issues in order, and only so do the matrix cores work during its softmax.  Same
        // arithmetic as the staged path.
        const u32x4_t kview = view_words(src.keys, (cached ? p.rot_rows : p.capacity) * uint32_t(HEAD_DIM * 2));
        const u32x4_t vview = view_words(p.values, p.capacity * uint32_t(HEAD_DIM * 2));
        const int uw = __builtin_amdgcn_readfirstlane(wave);
        const uint32_t lds = lds_address(L) + uint32_t(uw) * 4096u;
        // load t of wave w: rows 16w + 4t .. + 3, lane l the slot l % 16 of row 16w + 4t + l / 16
        const uint32_t lrow = uint32_t(16 * uw + (lane >> 4));
        const uint32_t vsrc = lrow * 256u + (uint32_t((lane & 15) ^ ((lane >> 4) << 2)) << 4);
        uint32_t ksrc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
            ksrc[t] = (lrow + uint32_t(4 * t)) * 256u + (uint32_t((lane & 15) ^ (lane >> 4) ^ (4 * t)) << 4);
        uint32_t vfirst = (klo + uint32_t(j0 * FK)) % p.capacity;  // ring slot of the next value tile's first key
        // Piece t of tile j's keys, and of the next value tile.  A tile whose 64 rows are
        // consecutive adds its first row as a scalar; in a block's last tile rows past khi take key
        // khi, and value rows wrap at the ring's end.  A tile past the part's end is its last
        // again (nobody reads that copy).
        auto request_k = [&](int j, auto piece) {
            constexpr int t = decltype(piece)::value;
            const uint32_t k0 = klo + uint32_t(min(j, j1 - 1) * FK);
            const uint32_t dst = lds + uint32_t((j - j0) & 1) * 16384u + uint32_t(t) * 1024u;
            if (k0 + uint32_t(FK - 1) <= khi) load_to_lds_untracked(kview, dst, ksrc[t], k0 * 256u);
            else load_to_lds_untracked(kview, dst, min(lrow + uint32_t(4 * t), khi - k0) * 256u + (ksrc[t] & 255u), k0 * 256u);
        };
        auto request_v = [&](int j, auto piece) {
            constexpr int t = decltype(piece)::value;
            const uint32_t k0 = klo + uint32_t(min(j, j1 - 1) * FK);
            const uint32_t dst = lds + 32768u + uint32_t((j - j0) & 1) * 16384u + uint32_t(t) * 1024u;
            if (k0 + uint32_t(FK - 1) <= khi && vfirst + uint32_t(FK - 1) < p.capacity) {
                load_to_lds_untracked(vview, dst, vsrc, vfirst * 256u + uint32_t(t) * 1024u);
            } else {
                const uint32_t slot = vfirst + min(lrow + uint32_t(4 * t), khi - k0);
                load_to_lds_untracked(vview, dst, min(slot, slot - p.capacity) * 256u + (vsrc & 255u), 0u);
            }
        };
        auto advance_v = [&](int j) {  // to tile j
            if (j < j1) vfirst += uint32_t(FK);
            vfirst = vfirst >= p.capacity ? vfirst - p.capacity : vfirst;
        };
        // S^T operand of row tile r, k-step s: key row 32r + col, dims 16s + 8 half .. + 8
        const uint32_t kbase = uint32_t(col * 256 + ((half ^ (col & 15)) << 4));
        auto kop = [&](int buf, int r, int s) {
            return as_bf16x8(*reinterpret_cast<const uint4*>(L + buf * 16384 + r * 8192 + (kbase ^ uint32_t(s << 5))));
        };
        // V^T operand of d-tile dt, k-step s: source lane sl = lane % 16 of 16-lane group g =
        // lane / 16 addresses keys 16s + 4(g / 2) + sl / 4 (and + 8), dims 32dt + 16(g % 2) +
        // 4(sl % 4) .. + 3; the transposing read hands lane j of the group element j % 4 of
        // source lane 4t + j / 4 as its element t: dim 32dt + 16(g % 2) + j of keys 16s + 4(g / 2)
        // + t (and + 8 + t), the rows of the P^T operand's k-step s
        typedef short short4_t __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) short4_t* tr_ptr_t;
        const int sl = lane & 15, grp = lane >> 4;
        const uint32_t vbase = uint32_t((4 * (grp >> 1) + (sl >> 2)) * 256 + ((sl >> 2) << 6) + 32 * (grp & 1) + 8 * (sl & 3));
        auto vop = [&](int buf, int dt, int s) {
            const uint8_t* at = L + 32768 + buf * 16384 + s * 4096 + (vbase ^ uint32_t(dt << 6));
            const short4_t x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)at);
            const short4_t x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)(at + 2048));
            bf16x8 a;
            __builtin_memcpy(&a, &x0, 8);
            __builtin_memcpy(reinterpret_cast<char*>(&a) + 8, &x1, 8);
            return a;
        };
        // Each wave waits for its own loads into LDS and its LDS reads, then the barrier: every
        // tile requested so far is in, and the buffers of the tile before are free.
        auto tiles_in = [&] {
            __asm__ volatile("" ::: "memory");
            wait_vmcnt_lds<0>();
            __builtin_amdgcn_s_barrier();
            __asm__ volatile("" ::: "memory");
        };
        // S^T product i (0..15) of the tile in buffer `buf`: k-step i / 2, row tile i % 2; its
        // operand was read four products ago
        bf16x8 kf[4];
        auto st_first = [&](int buf) {
#pragma unroll
            for (int i = 0; i < 4; ++i) kf[i] = kop(buf, i & 1, i >> 1);
        };
        auto st = [&](int buf, auto n, floatx16 (&acc)[2]) {
            constexpr int i = decltype(n)::value;
            const floatx16 zero = {};
            acc[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[i & 3], qf[i >> 1], i < 2 ? zero : acc[i & 1], 0, 0, 0);
            if constexpr (i + 4 < 16) kf[i & 3] = kop(buf, i & 1, (i + 4) >> 1);
        };
        auto fence = [] { __builtin_amdgcn_sched_barrier(0); };

        // Tile j (buffer B), whose scores are in sc; with NEXT the scores of tile j + 1 go to sn
        // (without SHORT, after the last tile: of stale keys, for nobody)
        auto tile = [&](int j, auto par, auto next, floatx16 (&sc)[2], floatx16 (&sn)[2]) {
            constexpr int B = decltype(par)::value;
            constexpr bool NEXT = decltype(next)::value;
            tiles_in();
            const uint32_t k0 = klo + uint32_t(j * FK);
            const bool edge = QSA || !(k0 + uint32_t(FK - 1) <= plo && (p.full || k0 + uint32_t(WINDOW - 1) >= khi));
            float mt = NEG_INF;
            if constexpr (NEXT) {
                advance_v(j + 1);
                st_first(B ^ 1);
            }
            // step n of sixteen: a product of S^T and, in the first eight, a request of a tile after
            auto beside = [&](auto n) {
                constexpr int i = decltype(n)::value;
                if constexpr (NEXT) {
                    if constexpr (i < 4) request_v(j + 1, std::integral_constant<int, i & 3>{});
                    else if constexpr (i < 8) request_k(j + 2, std::integral_constant<int, i & 3>{});
                    st(B ^ 1, n, sn);
                }
            };
            if (edge) {
                // QSA (global layers: k0 is a multiple of 64): the tile's 16 blocks b0 .. b0 + 15
                // are bits 0..15 of one bitmap word shifted by b0 % 32, read once per tile; blocks
                // at or past qcomplete are not tested
                uint32_t qbits = 0u;
                const uint32_t b0 = k0 >> 2;
                if (QSA && b0 < qcomplete) qbits = qmask[b0 >> 5] >> (b0 & 31) >> half;
                // the lane's keys are k0 + 4 half + c for constants c
                const int last = int(qpos - k0) - 4 * half, first = p.full ? -FK : last - (WINDOW - 1);
                const int open = int(qcomplete - b0) - half;
                static_for<0, 16>([&](auto n) {
                    beside(n);
#pragma unroll
                    for (int e = 2 * decltype(n)::value; e < 2 * decltype(n)::value + 2; ++e) {
                        const int r = e >> 4, q = e & 15, c = 32 * r + 8 * (q >> 2) + (q & 3), b = c >> 2;
                        bool vis = c <= last && c >= first;
                        if (QSA) vis = vis && (b >= open || ((qbits >> b) & 1u));
                        const float x = vis ? sc[r][q] * SCALE_LOG2E : NEG_INF;
                        sc[r][q] = x;
                        mt = fmaxf(mt, x);
                    }
                    fence();
                });
            } else {
                static_for<0, 16>([&](auto n) {
                    constexpr int r = decltype(n)::value >> 3, q = 2 * decltype(n)::value & 15;
                    beside(n);
                    sc[r][q] = sc[r][q] * SCALE_LOG2E;
                    sc[r][q + 1] = sc[r][q + 1] * SCALE_LOG2E;
                    mt = fmaxf(fmaxf(mt, sc[r][q]), sc[r][q + 1]);
                    fence();
                });
            }
            mt = fmaxf(mt, xor_lane<32>(mt));
            const float mn = fmaxf(m, mt);
            const float ms = mn == NEG_INF ? 0.0f : mn;  // nothing visible yet: every p is 0
            const float alpha = exp2_det(m - ms);
            ls *= alpha;
            m = mn;
            // alpha is exactly 1 where the running maximum did not move: the wave skips the
            // rescale when that holds in every lane (multiplying by 1 changes nothing)
            if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
                for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                    for (int i = 0; i < 16; ++i) oacc[dt][i] *= alpha;
            }
            // Quarter s: keys 16s + 4 half + {0..3} and 16s + 8 + 4 half + {0..3} as one k-step of
            // P.V; product n of a quarter: d-tiles 0, 1 with hi then lo, then 2, 3
            uint32_t hw[2][4], lw[2][4];
            bf16x8 vf[2][2];
            vf[0][0] = vop(B, 0, 0);
            vf[0][1] = vop(B, 1, 0);
            static_for<0, 20>([&](auto n) {
                constexpr int s = decltype(n)::value >> 2, k = decltype(n)::value & 3;
                if constexpr (s > 0) {
                    constexpr int h = k >> 1, g = (s - 1) & 1;
                    bf16x8 pw;
                    if constexpr (k & 1) {
                        pw = as_bf16x8(make_uint4(lw[g][0], lw[g][1], lw[g][2], lw[g][3]));
                    } else {
                        pw = as_bf16x8(make_uint4(hw[g][0], hw[g][1], hw[g][2], hw[g][3]));
                        if constexpr (h == 0) {  // the operands of the next two d-tiles
                            vf[1][0] = vop(B, 2, s - 1);
                            vf[1][1] = vop(B, 3, s - 1);
                        } else if constexpr (s < 4) {
                            vf[0][0] = vop(B, 0, s);
                            vf[0][1] = vop(B, 1, s);
                        }
                    }
                    oacc[2 * h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[h][0], pw, oacc[2 * h], 0, 0, 0);
                    oacc[2 * h + 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[h][1], pw, oacc[2 * h + 1], 0, 0, 0);
                }
                if constexpr (s < 4) {
                    constexpr int r = s >> 1, i = (s & 1) * 8 + 2 * k;
                    const float e0 = exp2_det(sc[r][i] - ms), e1 = exp2_det(sc[r][i + 1] - ms);
                    ls += e0;
                    ls += e1;
                    split_bf16_dot2(e0, e1, hw[s & 1][k], lw[s & 1][k]);
                }
                fence();
            });
        };
        floatx16 sa[2], sb[2];
        static_for<0, 4>([&](auto t) { request_k(j0, t); });
        static_for<0, 4>([&](auto t) { request_v(j0, t); });
        tiles_in();
        st_first(0);
        if (!SHORT || j0 + 1 < j1) static_for<0, 4>([&](auto t) { request_k(j0 + 1, t); });
        static_for<0, 16>([&](auto n) { st(0, n, sa); });
        if constexpr (!SHORT) {
            for (int j = j0; j < j1; j += 2) {
                tile(j, std::integral_constant<int, 0>{}, std::true_type{}, sa, sb);
                if (j + 1 < j1) tile(j + 1, std::integral_constant<int, 1>{}, std::true_type{}, sb, sa);
            }
        } else if (j0 + 1 < j1) {
            tile(j0, std::integral_constant<int, 0>{}, std::true_type{}, sa, sb);
            tile(j0 + 1, std::integral_constant<int, 1>{}, std::false_type{}, sb, sa);
        } else {
            tile(j0, std::integral_constant<int, 0>{}, std::false_type{}, sa, sb);
        }
        wait_vmcnt<0>();  // no wave ends with a load into LDS in flight
    }
    // O = O^T / l; element i of d-tile dt is dim 32dt + 8(i/4) + 4*half + i%4
    float lt = ls + xor_lane<32>(ls);
    if (!SHORT && parts > 1) {
        // Partial (m, l, unnormalised O^T) of this part; the last part to finish merges all
        // parts of the block in part order: M = max m_q, w_q = 2^(m_q - M),
        // O = sum O_q w_q / sum l_q w_q.  A lane writes its sixteen 16-byte pieces where the same
        // lane of the merging part reads them, whole lines per wave (in column order a part's
        // 64 KB were 2,048 partial lines: 152 -> 136 us for 2048 queries from position 2048), and
        // the merging part keeps its own in registers.
        const uint32_t nslots = uint32_t(p.blocks) * FLASH_PARTS;
        const __amdgpu_buffer_rsrc_t ov = buffer_view(p.part_o, nslots * (FT * HEADS) * HEAD_DIM * 4u);
        const __amdgpu_buffer_rsrc_t mv = buffer_view(p.part_ml, nslots * (FT * HEADS) * 8u);
        auto o_off = [&](int q, int i) { return (uint32_t(block * FLASH_PARTS + q) * 16u + uint32_t(i)) * 4096u + uint32_t(tid) * 16u; };
        auto ml_off = [&](int q) { return (uint32_t(block * FLASH_PARTS + q) * 128u + uint32_t(wave * 32 + col)) * 8u; };
#pragma unroll
        for (int i = 0; i < 16; ++i)
            buffer_store16_sc1(ov, o_off(part, i),
                               make_uint4(__float_as_uint(oacc[i >> 2][4 * (i & 3)]), __float_as_uint(oacc[i >> 2][4 * (i & 3) + 1]),
                                          __float_as_uint(oacc[i >> 2][4 * (i & 3) + 2]), __float_as_uint(oacc[i >> 2][4 * (i & 3) + 3])));
        if (half == 0) buffer_store8_sc1(mv, ml_off(part), make_uint2(__float_as_uint(m), __float_as_uint(lt)));
        wait_stores();
        __syncthreads();
        if (tid == 0) s_last = atomicAdd(p.tickets + block, 1u) == uint32_t(parts - 1);
        __syncthreads();
        if (!s_last) return;
        if (tid == 0) atomicExch(p.tickets + block, 0u);  // ready for the next launch
        // the other one or two parts, a before b, their outputs requested twelve pieces at a time
        constexpr int BATCH = 12;
        const int qa = part == 0 ? 1 : 0, qc = part == 2 ? 1 : 2;
        const bool three = parts == 3;
        const uint2 mla = buffer_load8_sc1(mv, ml_off(qa));
        const uint2 mlb = three ? buffer_load8_sc1(mv, ml_off(qc)) : make_uint2(__float_as_uint(NEG_INF), 0u);
        const float ma = __uint_as_float(mla.x), mb = __uint_as_float(mlb.x);
        const float M = fmaxf(fmaxf(m, ma), mb);
        const float w = exp2_det(m - M), wa = exp2_det(ma - M), wb = exp2_det(mb - M);
        const float la = __uint_as_float(mla.y) * wa, lb = __uint_as_float(mlb.y) * wb, lown = lt * w;
        // The sums in part order.  Without a third part its terms are +0 at the end, which change
        // nothing (a sum that starts from +0 is never -0).
        auto merge = [&](auto first, auto second, auto third) {
            lt = ((0.f + first(lown, la, lb)) + second(lown, la, lb)) + third(lown, la, lb);
            static_for<0, (16 + BATCH - 1) / BATCH>([&](auto batch) {
                constexpr int i0 = decltype(batch)::value * BATCH, n = i0 + BATCH < 16 ? BATCH : 16 - i0;
                uint4 va[n], vb[n];
#pragma unroll
                for (int i = 0; i < n; ++i) va[i] = buffer_load16_sc1(ov, o_off(qa, i0 + i));
#pragma unroll
                for (int i = 0; i < n; ++i) vb[i] = three ? buffer_load16_sc1(ov, o_off(qc, i0 + i)) : make_uint4(0, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < n; ++i) {
                    const uint32_t xa[4] = {va[i].x, va[i].y, va[i].z, va[i].w}, xb[4] = {vb[i].x, vb[i].y, vb[i].z, vb[i].w};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int dt = (i0 + i) >> 2, e = 4 * ((i0 + i) & 3) + k;
                        const float o = oacc[dt][e] * w, a = __uint_as_float(xa[k]) * wa, b = __uint_as_float(xb[k]) * wb;
                        oacc[dt][e] = ((0.f + first(o, a, b)) + second(o, a, b)) + third(o, a, b);
                    }
                }
            });
        };
        auto own = [](float o, float, float) { return o; };
        auto pa = [](float, float a, float) { return a; };
        auto pb = [](float, float, float b) { return b; };
        if (part == 0) merge(own, pa, pb);
        else if (part == 1) merge(pa, own, pb);
        else merge(pa, pb, own);
    }
    if (!qvalid) return;
    uint16_t* orow = p.out + size_t(tq) * ATTN + head * HEAD_DIM;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            uint32_t w[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint32_t a = bits(roundbf(oacc[dt][4 * g + 2 * k] / lt));
                const uint32_t b = bits(roundbf(oacc[dt][4 * g + 2 * k + 1] / lt));
                w[k] = (a & 0xffffu) | (b << 16);
            }
            *reinterpret_cast<uint2*>(orow + 32 * dt + 8 * g + 4 * half) = make_uint2(w[0], w[1]);
        }
}

// Workgroup w takes part w / blocks of query block blocks - 1 - w % blocks (consecutive
// workgroups, dealt round-robin to the XCDs, take different blocks; a block's parts share an
// XCD) and returns if the block has fewer parts.
template <bool QSA, bool DIRECT, bool SHORT>
__global__ __launch_bounds__(256, 2) void flash_prefill_kernel(const FlashParams p) {
    const int nqb = p.blocks;
    flash_prefill<QSA, DIRECT, SHORT>(p, nqb - 1 - int(blockIdx.x) % nqb, int(blockIdx.x) / nqb);
}

// Workgroup w takes the item the host's schedule ranks for it (qb << 2 | part).
template <bool QSA, bool DIRECT>
__global__ __launch_bounds__(256, 2) void flash_prefill_ranked_kernel(const FlashParams p, const FlashSchedule sched) {
    const uint32_t item = sched.item[blockIdx.x];
    flash_prefill<QSA, DIRECT, false>(p, int(item >> 2), int(item & 3u));
}

template <int BT, int BW, int WT, int NT, int NS>
void launch_gemm_dma(GemmEpilogue epi, const GemmParams& p, hipStream_t s) {
    const int cols = epi == GEMM_SWIGLU ? INTER / (BW / 2) : (p.m + BW - 1) / BW;
    const int rows = (p.tokens + BT - 1) / BT;
    const int per = (cols * rows + 7) / 8;
    const dim3 grid(8 * per), block(NT);
#define PLAMO_GEMM(EP) hipLaunchKernelGGL((gemm_dma_kernel<EP, BT, BW, WT, NT, NS>), grid, block, 0, s, p, cols, rows)
    constexpr int TW = BW / (NT / 64 / WT) / 32;  // 32-column blocks per wave
    if constexpr (TW % 2 == 0) {  // gate and up blocks pair inside a wave: the SwiGLU tile
        PLAMO_GEMM(GEMM_SWIGLU);
    } else {
        if (epi == GEMM_F32) PLAMO_GEMM(GEMM_F32);
        else if (epi == GEMM_BF16) PLAMO_GEMM(GEMM_BF16);
        else PLAMO_GEMM(GEMM_RAW);
    }
#undef PLAMO_GEMM
}

template <int BT, int BM, int WT, int WM, int NT, int H, int NS>
void launch_gemm_small(GemmEpilogue epi, const GemmParams& p, hipStream_t s) {
    const int cols = epi == GEMM_SWIGLU ? INTER / (BM / 2) : (p.m + BM - 1) / BM;
    const int rows = (p.tokens + BT - 1) / BT;
    const int per = (cols * rows + 7) / 8;
    const dim3 grid(8 * per), block(NT);
    // four outputs per store where every row of y starts on such a boundary; the same check
    // covers y itself, which may be a view with only its elements' alignment
    const uintptr_t y = epi == GEMM_BF16 ? reinterpret_cast<uintptr_t>(p.y16) : reinterpret_cast<uintptr_t>(p.y);
    const int wide = p.m % 4 == 0 && y % (epi == GEMM_BF16 ? 8 : 16) == 0;
#define PLAMO_GEMM(EP) hipLaunchKernelGGL((gemm_small_kernel<EP, BT, BM, WT, WM, NT, H, NS>), grid, block, 0, s, p, cols, rows, wide)
    if (epi == GEMM_F32) PLAMO_GEMM(GEMM_F32);
    else if (epi == GEMM_BF16) PLAMO_GEMM(GEMM_BF16);
    else PLAMO_GEMM(GEMM_RAW);
#undef PLAMO_GEMM
}

template <int BT, int BM, int WT, int WM, int NT, int H, int NS>
void launch_swiglu_small(const GemmParams& p, hipStream_t s) {
    const int cols = INTER / (BM / 2), rows = (p.tokens + BT - 1) / BT, per = (cols * rows + 7) / 8;
    const int wide = reinterpret_cast<uintptr_t>(p.y16) % 8 == 0;
    hipLaunchKernelGGL((gemm_small_kernel<GEMM_SWIGLU, BT, BM, WT, WM, NT, H, NS>), dim3(8 * per), dim3(NT), 0, s, p,
                       cols, rows, wide);
}

// CUs of the current device.
int device_cus() {
    thread_local int of = -1, cus = 0;
    int device = 0;
    PLAMO_HIP(hipGetDevice(&device));
    if (device != of) {
        PLAMO_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
        cus = std::max(cus, 1);
        of = device;
    }
    return cus;
}

// A tile of the GEMM kernels and the measured time of one round of it (us; every CU one tile).
struct GemmTile {
    int bt, bm;
    float us;
    bool k256;  // its stages are 256 deep
};
// The tile whose rounds over the CUs take least.  A call of few tokens thus takes the largest tiles
// that still fill the chip, or small ones down to 16 x 16: every CU reads (bt + bm) rows of k values
// however the tile is cut, so the smallest that fits one round is also the shortest.
// A round is counted as one tile per CU, and each as long as the first.  That is so for tiles of more
// than 80 KB of LDS (down at 256 and 512 of them: 64 x 48 21.4 and 41.4 us, 64 x 96 31.2 and 63.6).
// Of the smaller ones two fit on a CU, and their second round is charged more than it takes: 16 x 16
// 8.9 and 10.8 us, 16 x 32 11.3 and 14.7, 32 x 32 11.3 and 19.6; gate_up's 16 x 64 8.3 and 9.2, 32 x 64
// 8.4 and 10.3, 64 x 96 11.3 and 17.1.
template <size_t N>
int gemm_tile(const GemmTile (&tiles)[N], int cols, int tokens, int k) {
    const int cus = device_cus();
    int best = -1;
    float least = 0.f;
    for (size_t i = 0; i < N; ++i) {
        const GemmTile& t = tiles[i];
        if (t.k256 && k % 256 != 0) continue;
        const int64_t n = int64_t((cols + t.bm - 1) / t.bm) * ((tokens + t.bt - 1) / t.bt);
        const float us = float((n + cus - 1) / cus) * t.us;
        // of equal times the larger tile, in fewer rounds (qkv of 1,281 to 1,344 tokens: 128 x 128 in
        // one round 15.6 us, 96 x 64 in two 18.1)
        if (best < 0 || us <= least) best = int(i), least = us;
    }
    return best;
}

template <int BT, int BW, int WT, int NT>
void launch_gemm_packed(GemmEpilogue epi, const GemmParams& p, hipStream_t s) {
    const int cols = epi == GEMM_SWIGLU ? INTER / (BW / 2) : (p.m + BW - 1) / BW;
    const int rows = (p.tokens + BT - 1) / BT;
    const int per = (cols * rows + 7) / 8;
    const dim3 grid(8 * per), block(NT);
#define PLAMO_GEMM(PK, EP) hipLaunchKernelGGL((gemm_kernel<PK, EP, BT, BW, WT, NT>), grid, block, 0, s, p, cols, rows)
    if (epi == GEMM_F32) PLAMO_GEMM(true, GEMM_F32);
    else if (epi == GEMM_BF16) PLAMO_GEMM(true, GEMM_BF16);
    else if (epi == GEMM_RAW) PLAMO_GEMM(true, GEMM_RAW);
    else PLAMO_GEMM(true, GEMM_SWIGLU);
#undef PLAMO_GEMM
}

}  // namespace

void launch_gemm(bool packed, GemmEpilogue epi, const GemmParams& p, hipStream_t s) {
    if (p.k % 128 != 0 || p.tokens < 1 || p.m < 1 || (epi == GEMM_SWIGLU && p.m != 2 * INTER))
        throw Error(E_INVAL, "unsupported GEMM shape");
    // operand and output views take 32-bit byte offsets (rows of the last tile included)
    const uint64_t t_pad = uint64_t(p.tokens) + 256;
    if (t_pad * uint64_t(p.k) * 2 >= (1ull << 31) || uint64_t(p.m) * uint64_t(p.k) * 2 >= (1ull << 31) ||
        t_pad * uint64_t(p.m) * 4 >= (1ull << 31))
        throw Error(E_INVAL, "GEMM operands exceed 2 GiB");
    if (packed) {  // .p12 weights expanded in registers on the way to LDS
        if (p.tokens > 128 && (epi == GEMM_SWIGLU || p.m > 2048)) launch_gemm_packed<256, 128, 4, 512>(epi, p, s);
        else launch_gemm_packed<128, 128, 2, 256>(epi, p, s);
        return;
    }
    // Tile choice: measured round times, cold weights.  gate_up (1536 deep), before (256 x 128
    // and 128 x 128 tiles only) and now: 16 tokens 19.7 -> 9.1 us, 77 21.8 -> 12.1, 256 27.4 ->
    // 20.4, 400 25.4 -> 23.6, 1024 53 -> 41, 1500 81 -> 69.
    if (epi == GEMM_SWIGLU) {
        static constexpr GemmTile tiles[] = {{16, 64, 9.1f, false},    {32, 64, 9.8f, false},   {64, 64, 11.5f, false},
                                             {64, 96, 13.5f, false},   {128, 128, 19.5f, false}, {192, 128, 23.4f, false},
                                             {128, 192, 25.5f, false}, {256, 128, 28.2f, false},
                                             {256, 192, 43.5f, false}};
        switch (gemm_tile(tiles, 2 * INTER, p.tokens, p.k)) {
            case 0: return launch_swiglu_small<16, 64, 1, 2, 128, 2, 4>(p, s);
            case 1: return launch_swiglu_small<32, 64, 2, 2, 256, 2, 3>(p, s);
            case 2: return launch_swiglu_small<64, 64, 4, 2, 512, 2, 3>(p, s);
            case 3: return launch_swiglu_small<64, 96, 4, 1, 256, 1, 4>(p, s);
            case 4: return launch_swiglu_small<128, 128, 2, 4, 512, 1, 4>(p, s);
            case 5: return launch_swiglu_small<192, 128, 2, 4, 512, 1, 4>(p, s);
            case 6: return launch_swiglu_small<128, 192, 4, 2, 512, 1, 3>(p, s);
            case 7: return launch_gemm_dma<256, 128, 4, 512, 3>(epi, p, s);
            default: return launch_swiglu_small<256, 192, 4, 2, 512, 1, 2>(p, s);
        }
    }
    // The other projections; round times of down (6144 deep; the ratios hold at 1536 and 2048).
    // Before (128 x 96 and 128 x 192 tiles only) and now: down 16 tokens 36.9 -> 9.4 us, 77 43.4
    // -> 12.3, 300 38.9 -> 18.7, 1024 46 -> 35, 1500 48 -> 40.5; o 16 tokens 14.5 -> 4.6, 300 15.2
    // -> 7.9, 1024 17.1 -> 13.5; qkv 16 tokens 11.9 -> 4.2, 300 18.6 -> 8.1, 1024 19.7 -> 16.2.
    // A small tile's time is the time to fill its stages, (bt + bm) rows through the CU's vector
    // memory path: operands read a stage ahead, loads spread between the products, and
    // activations loaded into registers instead of LDS all measured the same or slower.
    static constexpr GemmTile tiles[] = {{16, 16, 9.4f, true},     {16, 16, 9.6f, false},   {32, 16, 10.5f, true},
                                         {16, 32, 12.2f, false},   {32, 32, 14.0f, false},  {64, 32, 18.0f, false},
                                         {64, 48, 22.0f, false},   {64, 64, 25.0f, false},  {96, 64, 28.0f, false},
                                         {128, 64, 37.0f, false},  {64, 96, 35.0f, false},  {96, 96, 40.0f, false},
                                         {128, 96, 49.0f, false},  {128, 128, 56.0f, false}, {128, 192, 74.0f, false}};
    switch (gemm_tile(tiles, p.m, p.tokens, p.k)) {
        case 0: return launch_gemm_small<16, 16, 1, 1, 256, 4, 4>(epi, p, s);
        case 1: return launch_gemm_small<16, 16, 1, 1, 256, 2, 8>(epi, p, s);
        case 2: return launch_gemm_small<32, 16, 2, 1, 256, 4, 4>(epi, p, s);
        case 3: return launch_gemm_small<16, 32, 1, 2, 256, 2, 6>(epi, p, s);
        case 4: return launch_gemm_small<32, 32, 2, 2, 256, 2, 4>(epi, p, s);
        case 5: return launch_gemm_small<64, 32, 4, 1, 256, 2, 4>(epi, p, s);
        case 6: return launch_gemm_small<64, 48, 4, 1, 256, 2, 4>(epi, p, s);
        case 7: return launch_gemm_small<64, 64, 4, 2, 512, 2, 3>(epi, p, s);
        case 8: return launch_gemm_small<96, 64, 2, 4, 512, 2, 3>(epi, p, s);
        case 9: return launch_gemm_small<128, 64, 4, 2, 512, 1, 4>(epi, p, s);
        case 10: return launch_gemm_small<64, 96, 4, 2, 512, 2, 3>(epi, p, s);
        case 11: return launch_gemm_small<96, 96, 2, 3, 384, 1, 4>(epi, p, s);
        case 12: return launch_gemm_dma<128, 96, 4, 256, 4>(epi, p, s);
        case 13: return launch_gemm_small<128, 128, 2, 4, 512, 1, 4>(epi, p, s);
        default: return launch_gemm_dma<128, 192, 4, 512, 3>(epi, p, s);
    }
}

void launch_rows_norm(const RowsNormParams& p, int tokens, hipStream_t s) {
    RowsNormParams q = p;
    q.tokens = tokens;
    hipLaunchKernelGGL(rows_norm_kernel, dim3((tokens + 3) / 4), dim3(256), 0, s, q);
}

void launch_gather_last(const uint16_t* a, const uint16_t* b, const PrefillSegments& seg, uint16_t* a_out, uint16_t* b_out,
                        hipStream_t s) {
    hipLaunchKernelGGL(gather_last_kernel, dim3(seg.n), dim3(HIDDEN / 8), 0, s, a, b, seg, a_out, b_out);
}

void launch_qk_prep(const QkPrepParams& p, hipStream_t s) {
    if (p.tokens < 1) return;
    if (!p.seg.valid()) throw Error(E_INVAL, "prefill: bad segments");
    hipLaunchKernelGGL(qk_prep_kernel, dim3(p.tokens), dim3(256), 0, s, p);
}

namespace {

// Workgroup order of a flash call whose items all fit on the GPU at once (its arithmetic does
// not depend on the order).  The items (query block, part) are ranked by their tile count,
// largest first (ties: later block, then lower part).  Two workgroups of this kernel fit on a
// CU, and workgroups w and w + CUs of a launch whose workgroups all start together share a
// CU, so workgroups CUs .. take the ranks from CUs on in reverse: the largest items share a CU
// with the smallest.  Measured on a 2048-token call from position 0 (504 items): the most
// tiles on one CU 23 -> 18, flash 66 -> 62 us.  Calls with more items than two per CU keep
// the default order (all parts of a block on one XCD): the ranked order measured 3 % slower
// on the later chunks of a 30,720-token prompt.
void flash_schedule(const FlashParams& p, FlashSchedule& sched) {
    // the last schedule of local and of global layers, per host thread
    thread_local struct {
        int cus = 0, tokens[PREFILL_SEGMENTS] = {-1};
        uint32_t p0 = 0;
        FlashSchedule sched{};
    } cache[2];
    int lengths[PREFILL_SEGMENTS] = {};
    for (int i = 0; i < p.seg.n; ++i) lengths[i] = p.seg.s[i].tokens;
    auto& c = cache[p.full ? 1 : 0];
    const int C = device_cus();
    if (c.cus != C || !std::equal(lengths, lengths + PREFILL_SEGMENTS, c.tokens) || c.p0 != p.p0) {
        struct Item {
            int tiles, qb, part;
        };
        Item items[FLASH_SCHEDULE_MAX];
        int n = 0;
        for (int qb = 0; qb < p.blocks; ++qb) {
            const PrefillSegment sg = p.seg.of_block(qb);
            const int tiles = flash_block_tiles(sg.tokens, p.p0, p.full, qb - sg.first_block), parts = flash_block_parts(tiles);
            for (int q = 0; q < parts; ++q) items[n++] = {(q + 1) * tiles / parts - q * tiles / parts, qb, q};
        }
        c.sched.n = 0;
        if (n <= 2 * C) {
            std::sort(items, items + n, [](const Item& a, const Item& b) {
                if (a.tiles != b.tiles) return a.tiles > b.tiles;
                if (a.qb != b.qb) return a.qb > b.qb;
                return a.part < b.part;
            });
            for (int w = 0; w < n; ++w) {
                const int rank = w < C ? w : C + (n - 1 - w);
                c.sched.item[w] = uint16_t((items[rank].qb << 2) | items[rank].part);
            }
            c.sched.n = uint32_t(n);
        }
        std::copy(lengths, lengths + PREFILL_SEGMENTS, c.tokens);
        c.p0 = p.p0;
        c.cus = C;
    }
    sched = c.sched;
}

}  // namespace

void launch_flash_prefill(const FlashParams& params, hipStream_t s) {
    FlashParams p = params;
    if (!p.seg.valid()) throw Error(E_INVAL, "prefill: bad segments");
    p.blocks = flash_blocks(p.seg);
    if (p.blocks < 1) return;
    if (p.blocks > 65536 / FLASH_PARTS) throw Error(E_INVAL, "flash prefill: too many tokens in one call");
    const bool qsa = p.full && p.qsa_mask;
    // keys straight into LDS when no block of the call rotates its keys: global layers, and
    // local layers whose keys all sit in the rotated-key cache (window base 0)
    uint32_t last = 0;
    for (int i = 0; i < p.seg.n; ++i) last = std::max(last, p.p0 + uint32_t(p.seg.s[i].tokens) - 1);
    const bool direct = p.capacity >= uint32_t(FK) &&
                        (p.full || (p.keys_rot != nullptr && last < p.rot_rows && last < uint32_t(WINDOW)));
    const dim3 block(256);
    // every block within two tiles of keys (key `last` is the last of them): one part each
    if (direct && last < uint32_t(2 * FK)) {
        const dim3 grid(uint32_t(p.blocks));
        if (qsa) hipLaunchKernelGGL((flash_prefill_kernel<true, true, true>), grid, block, 0, s, p);
        else hipLaunchKernelGGL((flash_prefill_kernel<false, true, true>), grid, block, 0, s, p);
        return;
    }
    FlashSchedule sched;
    sched.n = 0;
    if (p.blocks * FLASH_PARTS <= FLASH_SCHEDULE_MAX) flash_schedule(p, sched);
    if (sched.n) {
        // the schedule travels in the kernel arguments (1.5 KB): only the launches that use it
        const dim3 grid(sched.n);
#define PLAMO_FLASH(Q, D) hipLaunchKernelGGL((flash_prefill_ranked_kernel<Q, D>), grid, block, 0, s, p, sched)
        if (qsa) PLAMO_FLASH(true, true);
        else if (direct) PLAMO_FLASH(false, true);
        else PLAMO_FLASH(false, false);
#undef PLAMO_FLASH
    } else {
        const dim3 grid(uint32_t(p.blocks * FLASH_PARTS));
#define PLAMO_FLASH(Q, D) hipLaunchKernelGGL((flash_prefill_kernel<Q, D, false>), grid, block, 0, s, p)
        if (qsa) PLAMO_FLASH(true, true);
        else if (direct) PLAMO_FLASH(false, true);
        else PLAMO_FLASH(false, false);
#undef PLAMO_FLASH
    }
}

}  // namespace plamo
