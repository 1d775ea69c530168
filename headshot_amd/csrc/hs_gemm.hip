// Linear layers for gfx950 (replaces GpuContext::linear, engine/ops.rs:81-128,
// shaders/linear_wmma.wgsl and shaders/linear.wesl): out (M, N) = x (M, K)
// @ w (N, K)^T + bias (N, f32), with the epilogues the trunk's blocks apply
// to the result fused into the store (model/block.rs:150-176):
//   EPI_BIAS      out = f16(acc + bias)                       (qkv, linear)
//   EPI_GELU      out = f16(gelu(acc + bias))                 (fc1 + GELU)
//   EPI_LS        out = f16(res + gamma * f16(acc + bias))    (proj/fc2 +
//                                                 LayerScale + residual)
//   EPI_QKV       the fused q|k|v projection: f16(acc + bias), split into
//                 heads and written head-major, with QK-norm and RoPE
//                 applied to q and k (model/block.rs:128-146)
// so the activation between a GEMM and its elementwise op never crosses HBM.
//
// Fast path (f16, N % 256 == 0, K % kBK == 0): matrix-core GEMM. A workgroup
// computes one tile of out in a shape chosen by the tile count (256 x 256 down
// to 64 x 64, F16Tile), K in steps of kBK staged through a ring in LDS (the
// coming steps' tiles go straight from global memory into LDS with
// buffer_load_dwordx4 ... lds while the current one computes, with no
// registers in between). Both operands are K-contiguous rows (x rows, w rows),
// which is exactly the operand layout of v_mfma_f32_32x32x16_f16, so both come
// from LDS with 16-byte reads. Each wave owns 32, 96 or 128 rows x 64 columns
// and computes the transposed tile
// out^T = w x^T: its accumulators then hold, per lane, 4 consecutive output
// columns of one output row. The epilogue adds the bias (and applies GELU)
// there, stages the f16 results through LDS, and then streams whole rows:
// 16-byte reads of the residual and 16-byte writes of out. Rows past M are
// clamped on load and masked on store. The writes are non-temporal: every
// workgroup of a round stores its tile at about the same time, and streaming
// stores drain that burst faster than write-allocating ones (fc1 + GELU at
// S=32: 494 us against 523).
//
// f32 (N % 128 == 0, K % 32 == 0; every epilogue, with or without the LayerNorm
// prologue): each operand as three bf16 values on the bf16 matrix cores
// (gemm_split_kernel), or for few rows a kernel that splits K over its waves
// and streams the weights straight into registers (gemm_skinny_kernel).
//
// Generic path (the shapes neither covers): a tiled scalar kernel, f32
// accumulation in K order.
#include <math.h>

#include <initializer_list>
#include <mutex>
#include <type_traits>

#include "hs_common.hpp"

namespace hs {
namespace {

typedef f16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

enum Epi { EPI_BIAS = 0, EPI_GELU = 1, EPI_LS = 2, EPI_QKV = 3 };

// The q|k|v epilogue's outputs and parameters: out[0..2] head-major (S, H,
// T, 64) q, k, v; QK-norm weight / bias per q and k (null: none); RoPE
// tables (T - prefix, 64) (null: none).
struct QkvArgs {
    void* out[3];  // f16 or f32, as the product
    const float* nw[2];
    const float* nb[2];
    const float* sin_tab;
    const float* cos_tab;
    int seq, heads, prefix;
    float eps;
};

// The LayerNorm prologue (hs_linear_ln*): stats holds each x row's (mean,
// rsqrt(var + eps)) from hs_layernorm_stats, ln_w / ln_b the LayerNorm's
// affine parameters over the K input columns. The product reads each x
// element as hs_layernorm would have stored it.
struct LnArgs {
    const float* stats;
    const float* ln_w;
    const float* ln_b;
};

// ---------------------------------------------------------------------------
// matrix-core path

#ifndef HS_GEMM_XCD
#define HS_GEMM_XCD 1  // XCD-aware tile order
#endif
constexpr int kBK = 64;                  // K per LDS stage
constexpr int kRowChunks = kBK / 8;      // 16-byte chunks per LDS row
constexpr int kRowsPerInstr = 64 / kRowChunks;
constexpr int kRowsPer256B = 128 / kBK;  // LDS rows per 64-bank period
static_assert((kBK / 16) % 2 == 0, "operand register sets alternate within a stage");
// Epilogue staging: each wave's block of 64 columns as f16 rows of kEpiPitch
// halves (144 B: 16-byte aligned rows, spread over the banks).
constexpr int kEpiPitch = 64 + 8;

// A tile shape: WM x WN waves of 32 RB rows x 64 columns each, a ring of ST
// stages in LDS, the refill of a freed stage issued in SP parts.
//
// Stages are filled by buffer_load_dwordx4 ... lds (LDS-DMA): one wave
// instruction puts its 64 lanes' 16-byte chunks into 1 KiB of LDS in lane
// order, i.e. kRowsPerInstr unpadded rows. Lane L of instruction j supplies
// row kRowsPerInstr * j + L / kRowChunks at physical chunk L % kRowChunks,
// which holds logical chunk (L % kRowChunks) ^ swz(row), swz(row) = (row /
// kRowsPer256B) % kRowChunks: with that XOR swizzle the operand reads (16
// consecutive rows, one logical chunk) hit 16 distinct 16-byte bank groups.
// The buffer form (a descriptor in scalar registers, a per-lane offset fixed
// for the tile, the stage's column in the scalar offset) costs no vector
// instruction per load, and unlike the global (FLAT-encoded) form it lets
// the compiler wait for the operand reads of one k-slice with lgkmcnt(n)
// while the next slice's reads are in flight.
template <int WM, int WN, int RB_, int ST_, int SP_>
struct F16Tile {
    static constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
    static constexpr int kWN = WN, kRB = RB_, kST = ST_, kSP = SP_;
    static constexpr int kBM = 32 * RB_ * WM;  // output rows per workgroup
    static constexpr int kBN = 64 * WN;        // output columns per workgroup
    static constexpr int kXL = kBM * kBK / 8 / 64 / kWaves;  // stage loads per wave, x
    static constexpr int kWL = kBN * kBK / 8 / 64 / kWaves;  // w
    static_assert(kXL * 64 * kWaves == kBM * kBK / 8 && kWL * 64 * kWaves == kBN * kBK / 8, "stage split");
    struct Smem {
        f16 x[ST_][kBM * kBK];
        f16 w[ST_][kBN * kBK];
    };
    // With the LayerNorm prologue, x stages land in `raw` one stage ahead of
    // their use and are normalised from there into x[]: raw follows Smem.
    static constexpr size_t kRawBytes = size_t{2} * kBM * kBK;
    static constexpr int kEpiWave = 32 * RB_ * kEpiPitch;  // halves per wave
    static constexpr size_t smem_bytes(bool ln) {
        const size_t loop = sizeof(Smem) + (ln ? kRawBytes : 0);
        const size_t epi = size_t{2} * kWaves * kEpiWave;
        return loop > epi ? loop : epi;
    }
    // waves per SIMD that the LDS lets a CU hold
    static constexpr int kGroups = 160 * 1024 / static_cast<int>(sizeof(Smem));
    static constexpr int kWavesPerEu = kGroups * kWaves >= 8 ? kGroups * kWaves / 4 : 1;
};
using F16Big = F16Tile<2, 4, 4, 2, 1>;    // 256 x 256, 8 waves, one workgroup per CU
using F16Mid = F16Tile<2, 4, 3, 2, 1>;    // 192 x 256, 8 waves, one per CU
using F16Pair = F16Tile<4, 2, 1, 2, 1>;   // 128 x 128, 8 waves, two per CU
using F16Solo = F16Tile<4, 2, 1, 4, 4>;   // 128 x 128, 8 waves, one per CU, four stages
using F16Small = F16Tile<2, 1, 1, 4, 4>;  // 64 x 64, 2 waves, two per CU, four stages
static_assert(F16Big::smem_bytes(true) <= 160 * 1024, "gfx950 has 160 KiB of LDS per workgroup");

__device__ __forceinline__ h8 as_h8(u32x4 v) { return __builtin_bit_cast(h8, v); }

typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ int swz(int row) { return (row / kRowsPer256B) % kRowChunks; }

// Per-lane byte offsets of this wave's stage loads within the tile's x and
// w row blocks; x rows past M read row M - 1 (their outputs are masked).
template <typename P>
struct StageOffsets {
    uint32_t x[P::kXL];
    uint32_t w[P::kWL];
};

template <typename P>
__device__ __forceinline__ StageOffsets<P> stage_offsets(int64_t m0, int M, int K, int wave, int lane) {
    StageOffsets<P> o;
    const int prow = lane / kRowChunks, pc = lane % kRowChunks;
#pragma unroll
    for (int i = 0; i < P::kXL; i++) {
        const int row = kRowsPerInstr * (wave + P::kWaves * i) + prow;
        const int lrow = static_cast<int>(min(m0 + row, static_cast<int64_t>(M) - 1) - m0);
        o.x[i] = static_cast<uint32_t>(lrow * K * 2 + 16 * (pc ^ swz(row)));
    }
#pragma unroll
    for (int i = 0; i < P::kWL; i++) {
        const int row = kRowsPerInstr * (wave + P::kWaves * i) + prow;
        o.w[i] = static_cast<uint32_t>(row * K * 2 + 16 * (pc ^ swz(row)));
    }
    return o;
}

// One LDS-DMA wave instruction: each lane's 16 bytes at voff + koff of the
// buffer into the 1 KiB at dst, in lane order.
__device__ __forceinline__ void lds_load(f16* dst, __amdgpu_buffer_rsrc_t src, uint32_t voff, int koff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_void*)dst, 16, voff, koff, 0, 0);
}

// The LayerNorm prologue. Lane L of a wave normalises exactly the 16-byte
// pieces that its own x loads put into LDS: instruction i's piece, at
// halves (wave + kWaves i) * 512 + 8 L, is row kRowsPerInstr (wave + kWaves
// i) + L / kRowChunks of the tile, logical chunk lc = (L % kRowChunks) ^
// swz(row), and swz(row) does not depend on i. So a lane needs only its own
// loads to have landed (vmcnt, no barrier), its rows' statistics stay in
// registers for the whole product, and each stage's parameters are the 8
// columns 8 lc of that stage.
constexpr int kLnWaves = F16Big::kWaves;  // the prologue runs in F16Big tiles
constexpr int kLnRows = F16Big::kXL;     // x pieces per lane and stage
static_assert((kRowsPerInstr * kLnWaves / kRowsPer256B) % kRowChunks == 0,
              "a lane's x pieces share one logical chunk");
constexpr int kLnParamLoads = 4;            // 16-byte loads of ln_w / ln_b per stage
#ifndef HS_GEMM_LN_SLICES
#define HS_GEMM_LN_SLICES 2  // k slices of a step over which the next stage is normalised
#endif
#ifndef HS_GEMM_LN_FIRST
#define HS_GEMM_LN_FIRST 1  // the first of those slices (the pieces are read at slice 0)
#endif
constexpr int kLnSlices = HS_GEMM_LN_SLICES;
constexpr int kLnFirst = HS_GEMM_LN_FIRST;
static_assert(kLnRows % kLnSlices == 0 && kLnFirst >= 0 && kLnFirst + kLnSlices < kBK / 16,
              "LayerNorm slices: the next stage's parameters load in a later slice");

struct LnLane {
    f32x2 st[kLnRows];  // (mean, rstd) of the lane's rows
    int col;            // first column of the lane's chunk within a stage
};

__device__ __forceinline__ LnLane ln_lane(const LnArgs& la, int64_t m0, int M, int wave, int lane) {
    LnLane ll;
#pragma unroll
    for (int i = 0; i < kLnRows; i++) {
        const int row = kRowsPerInstr * (wave + kLnWaves * i) + lane / kRowChunks;
        // rows past M were loaded from row M - 1 and are normalised with its
        // statistics (their products are masked)
        const int64_t r = min(m0 + row, static_cast<int64_t>(M) - 1);
        ll.st[i] = *reinterpret_cast<const f32x2*>(la.stats + 2 * r);
    }
    ll.col = 8 * ((lane % kRowChunks) ^ swz(kRowsPerInstr * wave + lane / kRowChunks));
    return ll;
}

// The LayerNorm parameters of the lane's 8 columns of the stage at column k0.
__device__ __forceinline__ void ln_params(const LnArgs& la, const LnLane& ll, int k0,
                                          float4 (&gb)[kLnParamLoads]) {
    const int c = k0 + ll.col;
    gb[0] = ld_f32x4(la.ln_w + c), gb[1] = ld_f32x4(la.ln_w + c + 4);
    gb[2] = ld_f32x4(la.ln_b + c), gb[3] = ld_f32x4(la.ln_b + c + 4);
}

// Halves offset of the lane's piece i within an x stage.
__device__ __forceinline__ int ln_off(int i, int wave, int lane) {
    return (wave + kLnWaves * i) * 512 + 8 * lane;
}

// One normalised piece: the 8 f16 values of v, with the row's (mean, rstd)
// and the lane's column parameters gb (ln_w then ln_b), rounded to f16 as
// hs_layernorm stores them.
__device__ __forceinline__ u32x4 ln_piece(u32x4 v, f32x2 st, const float4 (&gb)[kLnParamLoads]) {
    const float g[8] = {gb[0].x, gb[0].y, gb[0].z, gb[0].w, gb[1].x, gb[1].y, gb[1].z, gb[1].w};
    const float b[8] = {gb[2].x, gb[2].y, gb[2].z, gb[2].w, gb[3].x, gb[3].y, gb[3].z, gb[3].w};
    // x - mean as x * 1 - mean, a mixed-precision multiply-add on the f16
    // half itself: the same value without the conversion
    float one = 1.0f;
    asm("" : "+s"(one));
    const float neg = -st[0];
    float f[8];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const f16x2 h = u2h2(v[j]);
        f[2 * j] = as_f32(fmaf(fmaf(static_cast<float>(h.x), one, neg) * st[1], g[2 * j], b[2 * j]));
        f[2 * j + 1] = as_f32(fmaf(fmaf(static_cast<float>(h.y), one, neg) * st[1], g[2 * j + 1], b[2 * j + 1]));
    }
    return pack(f, f16{});
}

// Normalises all of the lane's pieces of the stage in `raw` into `dst`.
__device__ __forceinline__ void ln_stage(const f16* raw, f16* dst, const LnLane& ll,
                                         const float4 (&gb)[kLnParamLoads], int wave, int lane) {
#pragma unroll
    for (int i = 0; i < kLnRows; i++)
        st16(dst + ln_off(i, wave, lane), ln_piece(ld16(raw + ln_off(i, wave, lane)), ll.st[i], gb));
}

// Buffer descriptor word 3 for raw (unstructured, stride 0) buffers on gfx950.
constexpr int kRawBufferFlags = 0x00020000;

// Operand read: logical chunk k of LDS row `row` (rows of kBK halves).
__device__ __forceinline__ h8 ld_op(const f16* buf, int row, int k) {
    return as_h8(ld16(buf + row * kBK + 8 * (k ^ swz(row))));
}

__device__ __forceinline__ uint32_t pk_f16(float a, float b) {
    f16x2 h;
    h.x = static_cast<f16>(a), h.y = static_cast<f16>(b);
    return h22u(h);
}

// Phase 2 of the q|k|v epilogue: the wave's staged block is `rows` token rows
// of one head of q, k or v (its 64 columns). 8 lanes per row hold the head
// vector in the lane layout of qk_norm_rope_vec (the QK-norm / RoPE fused
// op's), so each head vector is normalised, rotated and rounded by the same
// code as there; each row's 128 bytes go to (frame, head, token) of the
// head-major output.
__device__ __forceinline__ void qkv_heads_out(const f16* stage, const QkvArgs& qa, int64_t row0,
                                              int M, int64_t col, int lane, int rows) {
    const int hd = qa.heads * 64;
    const int which = static_cast<int>(col / hd);            // 0 q, 1 k, 2 v: wave-uniform
    const int head = static_cast<int>(col - int64_t{which} * hd) / 64;
    const int piece = lane & 7;
    const bool upper = piece >= 4;
    const int ch = upper ? 32 + (7 - piece) * 8 : piece * 8;
    const float* nw = which < 2 ? qa.nw[which] : nullptr;
    const float* nb = which < 2 ? qa.nb[which] : nullptr;
    const bool norm = nw != nullptr;
    const bool rope = which < 2 && qa.sin_tab != nullptr;
    float wr[8], br[8];
    if (norm) {
        const float4 w0 = ld_f32x4(nw + ch), w1 = ld_f32x4(nw + ch + 4);
        const float4 b0 = ld_f32x4(nb + ch), b1 = ld_f32x4(nb + ch + 4);
        wr[0] = w0.x, wr[1] = w0.y, wr[2] = w0.z, wr[3] = w0.w;
        wr[4] = w1.x, wr[5] = w1.y, wr[6] = w1.z, wr[7] = w1.w;
        br[0] = b0.x, br[1] = b0.y, br[2] = b0.z, br[3] = b0.w;
        br[4] = b1.x, br[5] = b1.y, br[6] = b1.z, br[7] = b1.w;
    }
    f16* obase = static_cast<f16*>(qa.out[which]) + static_cast<int64_t>(head) * qa.seq * 64 + ch;
    const float sg = upper ? 1.0f : -1.0f;
    // this lane's row: token m = s * seq + t (m < 2^31), advanced by 8 rows
    // per step
    int64_t m = row0 + (lane >> 3);
    uint32_t s = static_cast<uint32_t>(m) / static_cast<uint32_t>(qa.seq);
    int t = static_cast<int>(static_cast<uint32_t>(m) - s * static_cast<uint32_t>(qa.seq));
    for (int rr = 0; rr < rows; rr += 8) {
        if (m >= M) break;  // rows grow with rr: the rest are past M too
        float f[8];
        unpack(ld16(stage + (rr + (lane >> 3)) * kEpiPitch + ch), f, f16{});
        const bool rot = rope && t >= qa.prefix;  // the same for the row's 8 lanes
        float cs[8], sn[8];
        if (rot) {
            const int64_t trow = static_cast<int64_t>(t - qa.prefix) * 64 + ch;
            const float4 c0 = ld_f32x4(qa.cos_tab + trow), c1 = ld_f32x4(qa.cos_tab + trow + 4);
            const float4 s0 = ld_f32x4(qa.sin_tab + trow), s1 = ld_f32x4(qa.sin_tab + trow + 4);
            cs[0] = c0.x, cs[1] = c0.y, cs[2] = c0.z, cs[3] = c0.w;
            cs[4] = c1.x, cs[5] = c1.y, cs[6] = c1.z, cs[7] = c1.w;
            sn[0] = sg * s0.x, sn[1] = sg * s0.y, sn[2] = sg * s0.z, sn[3] = sg * s0.w;
            sn[4] = sg * s1.x, sn[5] = sg * s1.y, sn[6] = sg * s1.z, sn[7] = sg * s1.w;
        }
        if (norm)
            qk_norm_rope_vec<f16, 8, true>(f, wr, br, qa.eps, rot, cs, sn);
        else
            qk_norm_rope_vec<f16, 8, false>(f, wr, br, qa.eps, rot, cs, sn);
        st16_nt(obase + (static_cast<int64_t>(s) * qa.heads * qa.seq + t) * 64, pack(f, f16{}));
        m += 8;
        t += 8;
        while (t >= qa.seq) t -= qa.seq, s++;
    }
}

// Grid: tiles_m * tiles_n workgroups, column tiles fastest, so workgroups
// running together share their x rows.
template <int EPI, typename P, bool LN>
__global__ __launch_bounds__(P::kThreads, P::kWavesPerEu) void gemm_f16_kernel(
    const f16* __restrict__ x, const f16* __restrict__ w, const float* __restrict__ bias,
    const float* __restrict__ gamma, const f16* res, f16* out, int M, int N, int K,
    int tiles_n, int ntiles, QkvArgs qa, LnArgs la) {
    static_assert(!LN || std::is_same_v<P, F16Big>, "the LayerNorm prologue runs in F16Big tiles");
    constexpr int kRB = P::kRB, kST = P::kST, kBM = P::kBM, kBN = P::kBN;
    __shared__ __align__(16) unsigned char smem_raw[P::smem_bytes(LN)];
    typename P::Smem& sm = *reinterpret_cast<typename P::Smem*>(smem_raw);
    f16* const raw = reinterpret_cast<f16*>(smem_raw + sizeof(typename P::Smem));  // LN only
    const int tid = threadIdx.x;
    const int lane = lane_id();
    const int wave = tid >> 6;
    const int l32 = lane & 31, hh = lane >> 5;
#if HS_GEMM_XCD
    // Workgroup b runs on XCD b % 8; XCD x takes the contiguous tile range
    // [x * per, (x + 1) * per), so the column tiles of one row tile (which
    // share its x rows) run on one XCD and its L2. The grid is padded to a
    // multiple of 8 workgroups.
    const int per = static_cast<int>(gridDim.x / 8);
    const int tile = static_cast<int>(blockIdx.x % 8) * per + static_cast<int>(blockIdx.x / 8);
    if (tile >= ntiles) return;  // padding, before any barrier
#else
    const int tile = static_cast<int>(blockIdx.x);
#endif
    const int64_t m0 = static_cast<int64_t>(tile / tiles_n) * kBM;
    const int64_t n0 = static_cast<int64_t>(tile % tiles_n) * kBN;
    const int wm = (wave / P::kWN) * (32 * kRB);  // wave's rows within the tile
    const int wn = (wave % P::kWN) * 64;   // wave's columns within the tile

    // acc[a][b]: out^T block of columns wn + 32 a .. + 32 (MFMA rows) and
    // rows wm + 32 b .. + 32 (MFMA columns); register r of lane (l32, hh)
    // is column 8 (r / 4) + 4 hh + r % 4, row l32 of the block.
    f32x16 acc[2][kRB];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < kRB; b++) acc[a][b] = f32x16{};

    const int nsteps = K / kBK;
    const int wv = wave_in_block();
    const StageOffsets<P> so = stage_offsets<P>(m0, M, K, wv, lane);
    const int xrows = static_cast<int>(min(static_cast<int64_t>(kBM), M - m0));
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<f16*>(x + m0 * K), 0, xrows * K * 2, kRawBufferFlags);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<f16*>(w + n0 * K), 0, kBN * K * 2, kRawBufferFlags);
    // Issue this wave's LDS-DMA loads of one stage's x (or w) rows into dst;
    // koff = the stage's first column, in bytes.
    auto issue_x = [&](f16* dst, int koff) {
#pragma unroll
        for (int i = 0; i < P::kXL; i++)
            lds_load(dst + (wv + P::kWaves * i) * 512, xr, so.x[i], koff);
    };
    auto issue_w = [&](f16* dst, int koff) {
#pragma unroll
        for (int i = 0; i < P::kWL; i++)
            lds_load(dst + (wv + P::kWaves * i) * 512, wr, so.w[i], koff);
    };
    // Loads [from, to) of a stage's kL per wave, x first.
    constexpr int kL = P::kXL + P::kWL, kPart = kL / P::kSP;
    static_assert(kPart * P::kSP == kL && P::kSP <= kBK / 16, "a stage's loads in equal parts, one per slice");
    auto issue_part = [&](int buf, int koff, int from, int to) {
#pragma unroll
        for (int i = 0; i < kL; i++) {
            if (i < from || i >= to) continue;
            if (i < P::kXL)
                lds_load(sm.x[buf] + (wv + P::kWaves * i) * 512, xr, so.x[i < P::kXL ? i : 0], koff);
            else
                lds_load(sm.w[buf] + (wv + P::kWaves * (i - P::kXL)) * 512, wr, so.w[i < P::kXL ? 0 : i - P::kXL], koff);
        }
    };
    // Both buffers start filled (stages 0 and 1). The waits below are
    // explicit: vmcnt counts this wave's loads, which complete in order, and
    // the barrier then covers every wave's.
    //
    // With the LayerNorm prologue, stage s's x lands in raw during step s - 2
    // (its parameters loaded just before it) and is normalised into x[s & 1]
    // by its own lanes during step s - 1, beside that step's multiplies; w
    // keeps the schedule above. Per wave, in issue order: params(s + 2),
    // x(s + 2) in the middle of step s, w(s + 2) after its closing barrier.
    constexpr int kXL = P::kXL, kWL = P::kWL;
    LnLane ll;
    float4 gb[kLnParamLoads];
    if constexpr (LN) {
        ll = ln_lane(la, m0, M, wv, lane);
        ln_params(la, ll, 0, gb);
        issue_x(raw, 0);
        issue_w(sm.w[0], 0);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kWL) : "memory");  // params(0), x(0)
        ln_stage(raw, sm.x[0], ll, gb, wv, lane);
        if (nsteps > 1) {
            ln_params(la, ll, kBK, gb);
            issue_x(raw, 2 * kBK);
            issue_w(sm.w[1], 2 * kBK);
            // w(0) landed; x[0]'s normalised pieces written
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLnParamLoads + kXL + kWL)
                         : "memory");
        } else {
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
    } else {
#pragma unroll
        for (int i = 0; i + 1 < kST; i++)
            if (i < nsteps) issue_part(i, 2 * i * kBK, 0, kL);
        if (kST - 1 < nsteps) issue_part(kST - 1, 2 * (kST - 1) * kBK, 0, kPart);
        if (nsteps >= kST)
            asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((kST - 2) * kL + kPart) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    }
    // Operand registers in two sets: the next 16-wide k slice is read from
    // LDS while the current one multiplies, across stage boundaries too.
    constexpr int kSl = kBK / 16;
    h8 A[2][2], B[2][kRB];
    auto read_slice = [&](int set, int buf, int ks) {
        const int kc = 2 * ks + hh;
#pragma unroll
        for (int a = 0; a < 2; a++) A[set][a] = ld_op(sm.w[buf], wn + 32 * a + l32, kc);
#pragma unroll
        for (int b = 0; b < kRB; b++) B[set][b] = ld_op(sm.x[buf], wm + 32 * b + l32, kc);
    };
    read_slice(0, 0, 0);
    if constexpr (LN) {
        // One step of the product with the prologue: the multiplies of stage
        // s and, beside them, NORM: stage s + 1's LayerNorm from raw into
        // x[cur ^ 1] (last read in step s - 1, before the barrier that
        // closed it), ISSUE: the loads of stage s + 2. The flags are
        // compile-time, so each step is one basic block in which the
        // scheduler can place the LayerNorm's vector work between the
        // multiplies. The lane's kLnRows pieces are read at slice 0 and
        // normalised over the first kLnSlices slices; raw is refilled at
        // slice 1, once the pieces are in registers, and the next stage's
        // parameters load at slice kLnSlices, once these are used.
        auto step = [&](int s, auto norm_c, auto issue_c) {
            constexpr bool NORM = decltype(norm_c)::value, ISSUE = decltype(issue_c)::value;
            const int cur = s & 1;
            u32x4 rw[kLnRows];
#pragma unroll
            for (int ks = 0; ks < kBK / 16; ks++) {
                const int p = ks & 1;  // kBK / 16 is even: set 0 holds slice 0 of every stage
                if constexpr (ISSUE) {
                    if (ks == 1) {
                        // the lane's raw pieces (read at slice 0) are in
                        // registers: refill raw with x(s + 2)
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        issue_x(raw, 2 * (s + 2) * kBK);
                    }
                }
                if (ks + 1 < kBK / 16) {
                    const int kc = 2 * (ks + 1) + hh;
#pragma unroll
                    for (int a = 0; a < 2; a++) A[p ^ 1][a] = ld_op(sm.w[cur], wn + 32 * a + l32, kc);
#pragma unroll
                    for (int b = 0; b < kRB; b++) B[p ^ 1][b] = ld_op(sm.x[cur], wm + 32 * b + l32, kc);
                }
                if constexpr (NORM) {
                    if (ks == 0) {
                        // params(s + 1), x(s + 1) landed; w(s + 1) may be in flight
                        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kWL) : "memory");
#pragma unroll
                        for (int i = 0; i < kLnRows; i++) rw[i] = ld16(raw + ln_off(i, wv, lane));
                    }
                    if (ks >= kLnFirst && ks < kLnFirst + kLnSlices) {
                        constexpr int per = kLnRows / kLnSlices;
#pragma unroll
                        for (int i = (ks - kLnFirst) * per; i < (ks - kLnFirst + 1) * per; i++)
                            st16(sm.x[cur ^ 1] + ln_off(i, wv, lane), ln_piece(rw[i], ll.st[i], gb));
                    }
                    if constexpr (ISSUE) {
                        if (ks == kLnFirst + kLnSlices) ln_params(la, ll, (s + 2) * kBK, gb);
                    }
                }
                if (ks + 1 == kBK / 16) {
                    // every wave's reads of stage s are done; w(s + 1) and
                    // the normalised x(s + 1) have landed (params(s + 2) and
                    // x(s + 2) may be in flight)
                    if constexpr (ISSUE)
                        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLnParamLoads + kXL)
                                     : "memory");
                    else
                        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    if constexpr (NORM) read_slice(p ^ 1, cur ^ 1, 0);
                    // w[cur] is free: refill it with stage s + 2, behind the
                    // reads and between the multiplies
                    if constexpr (ISSUE) issue_w(sm.w[cur], 2 * (s + 2) * kBK);
                }
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int b = 0; b < kRB; b++)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[p][a], B[p][b], acc[a][b], 0, 0, 0);
                if constexpr (NORM) {
                    // the compiler's own order: groups that forced the
                    // LayerNorm's vector work between the multiplies were
                    // slower (a 21x37 frame block of 16: 513 us against 502)
                } else {
                    __builtin_amdgcn_sched_group_barrier(0x100, 6, 0);  // LDS reads
                    __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);  // MFMAs
                }
            }
        };
        int s = 0;
        for (; s + 2 < nsteps; s++) step(s, std::true_type{}, std::true_type{});
        if (s + 1 < nsteps) step(s++, std::true_type{}, std::false_type{});
        step(s, std::false_type{}, std::false_type{});
    } else {
        // One stage's multiplies. The refill of a freed buffer goes out behind
        // the next slice's operand reads and between multiplies (ahead of
        // the reads, its burst kept them waiting: fc1 at S=32 442 us against
        // 414): part 0 behind the barrier that frees the buffer, parts 1 .. in
        // the next step's slices. MORE: parts 1 .. of stage s + kST - 1 are
        // issued; NEXT: part 0 of stage s + kST is.
        int cur = 0;
        auto step = [&](int s, auto more_c, auto next_c) {
            constexpr bool MORE = decltype(more_c)::value, NEXT = decltype(next_c)::value;
            const int nxt = cur + 1 == kST ? 0 : cur + 1;
            const int prv = cur == 0 ? kST - 1 : cur - 1;
#pragma unroll
            for (int ks = 0; ks < kSl; ks++) {
                const int p = ks & 1;
                int loads = 0;
                if (ks + 1 < kSl) {
                    read_slice(p ^ 1, cur, ks + 1);
                    if (MORE && ks + 1 < P::kSP) {
                        issue_part(prv, 2 * (s + kST - 1) * kBK, (ks + 1) * kPart, (ks + 2) * kPart);
                        loads = kPart;
                    }
                } else {
                    // every wave's reads of stage s are done and stage s + 1
                    // has landed (stages s + 2 .. s + kST - 1 may be in flight)
                    if constexpr (NEXT || MORE)
                        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((kST - 2) * kL) : "memory");
                    else
                        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    read_slice(p ^ 1, nxt, 0);  // (past the last stage: stale, not used)
                    if constexpr (NEXT) {
                        issue_part(cur, 2 * (s + kST) * kBK, 0, kPart);
                        loads = kPart;
                    }
                }
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int b = 0; b < kRB; b++)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[p][a], B[p][b], acc[a][b], 0, 0, 0);
                // the reads ahead of the multiplies, the loads between them
                __builtin_amdgcn_sched_group_barrier(0x100, 2 + kRB, 0);  // LDS reads
                if (loads) {
                    constexpr int per = (kPart + 2 * kRB - 1) / (2 * kRB);
#pragma unroll
                    for (int q = 0; q < 2 * kRB; q++) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // an MFMA
                        __builtin_amdgcn_sched_group_barrier(0x010, per, 0);  // loads
                    }
                } else {
                    __builtin_amdgcn_sched_group_barrier(0x008, 2 * kRB, 0);  // MFMAs
                }
            }
            cur = nxt;
        };
        int s = 0;
        for (; s + kST < nsteps; s++) step(s, std::true_type{}, std::true_type{});
        if (s + kST == nsteps) step(s++, std::true_type{}, std::false_type{});
        for (; s < nsteps; s++) step(s, std::false_type{}, std::false_type{});
    }

    // Epilogue, in two phases so that global memory sees whole rows.
    // 1. Each lane turns its accumulators (row l32 of block b, columns
    //    32 a + 8 r4 + 4 hh .. + 4) into the linear's stored value,
    //    f16(acc + bias) (for GELU: f16(gelu(acc + bias))), and writes it
    //    to the wave's staging block in LDS (free once every wave has left
    //    the main loop).
    f16* stage = reinterpret_cast<f16*>(smem_raw) + wave * P::kEpiWave;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) {
            const int cl = 32 * a + 8 * r4 + 4 * hh;  // column within the wave's block
            const float4 bv = bias ? ld_f32x4(bias + n0 + wn + cl) : float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int b = 0; b < kRB; b++) {
                float v[4];
                v[0] = acc[a][b][4 * r4] + bv.x, v[1] = acc[a][b][4 * r4 + 1] + bv.y;
                v[2] = acc[a][b][4 * r4 + 2] + bv.z, v[3] = acc[a][b][4 * r4 + 3] + bv.w;
                if constexpr (EPI == EPI_GELU) {
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = gelu_f(v[e]);
                }
                u32x2 o;
                o[0] = pk_f16(v[0], v[1]), o[1] = pk_f16(v[2], v[3]);
                *reinterpret_cast<u32x2*>(stage + (32 * b + l32) * kEpiPitch + cl) = o;
            }
        }
    // only this wave reads its block back: a wave-level fence suffices
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if constexpr (EPI == EPI_QKV) {
        qkv_heads_out(stage, qa, m0 + wm, M, n0 + wn, lane, 32 * kRB);
        return;
    }
    // 2. 8 lanes per 128-byte row piece, 8 rows per instruction: 16-byte
    //    loads of the staged values (and of res), 16-byte stores of out.
    const int c8 = 8 * (lane & 7);
    const int64_t n = n0 + wn + c8;
    float4 g0 = {0.0f, 0.0f, 0.0f, 0.0f}, g1 = g0;
    if constexpr (EPI == EPI_LS) g0 = ld_f32x4(gamma + n), g1 = ld_f32x4(gamma + n + 4);
#pragma unroll 4
    for (int rr = 0; rr < 32 * kRB; rr += 8) {
        const int rl = rr + (lane >> 3);
        const int64_t m = m0 + wm + rl;
        if (m >= M) break;  // rows grow with rr: the rest are past M too
        u32x4 v = ld16(stage + rl * kEpiPitch + c8);
        if constexpr (EPI == EPI_LS) {
            // res + gamma * x, x the linear's stored (f16) value
            const u32x4 r = ld16(res + m * N + n);
            const float gg[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const f16x2 xv = u2h2(v[q]), rv = u2h2(r[q]);
                v[q] = pk_f16(fmaf(gg[2 * q], static_cast<float>(xv.x), static_cast<float>(rv.x)),
                              fmaf(gg[2 * q + 1], static_cast<float>(xv.y), static_cast<float>(rv.y)));
            }
        }
        st16_nt(out + m * N + n, v);
    }
}

// ---------------------------------------------------------------------------
// f32 products: shared pieces

// The f32 q|k|v epilogue's staging: each wave's block (32 kRB token rows x
// one head's 64 columns, acc + bias) in rows of kQkvPitch floats (16-byte
// aligned, 4 banks apart), in the LDS the stages used.
constexpr int kQkvPitch = 68;
// The f32 q|k|v epilogue's second phase: the wave's staged block is `rows`
// token rows of one head of q, k or v. 16 lanes per row hold the head
// vector in the lane layout of the standalone f32 QK-norm / RoPE op (piece
// p < 8: channels 4 p .. + 4; p >= 8: 32 + 4 (15 - p) .. + 4), so each head
// vector is normalised and rotated by the same code as there, and each
// row's 256 bytes go to (frame, head, token) of the head-major output.
__device__ __forceinline__ void qkv_heads_out_f32(const float* stage, const QkvArgs& qa, int64_t row0,
                                                  int M, int64_t col, int lane, int rows) {
    const int hd = qa.heads * 64;
    const int which = static_cast<int>(col / hd);  // 0 q, 1 k, 2 v: wave-uniform
    const int head = static_cast<int>(col - int64_t{which} * hd) / 64;
    const int piece = lane & 15;
    const bool upper = piece >= 8;
    const int ch = upper ? 32 + (15 - piece) * 4 : piece * 4;
    const float* nw = which < 2 ? qa.nw[which] : nullptr;
    const float* nb = which < 2 ? qa.nb[which] : nullptr;
    const bool norm = nw != nullptr;
    const bool rope = which < 2 && qa.sin_tab != nullptr;
    float wr[4] = {0.0f, 0.0f, 0.0f, 0.0f}, br[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (norm) {
        const float4 w0 = ld_f32x4(nw + ch), b0 = ld_f32x4(nb + ch);
        wr[0] = w0.x, wr[1] = w0.y, wr[2] = w0.z, wr[3] = w0.w;
        br[0] = b0.x, br[1] = b0.y, br[2] = b0.z, br[3] = b0.w;
    }
    float* obase = static_cast<float*>(qa.out[which]) + static_cast<int64_t>(head) * qa.seq * 64 + ch;
    const float sg = upper ? 1.0f : -1.0f;
    // this lane's row: token m = s * seq + t (m < 2^31), advanced by 4 rows
    // per step
    int64_t m = row0 + (lane >> 4);
    uint32_t s = static_cast<uint32_t>(m) / static_cast<uint32_t>(qa.seq);
    int t = static_cast<int>(static_cast<uint32_t>(m) - s * static_cast<uint32_t>(qa.seq));
    for (int rr = 0; rr < rows; rr += 4) {
        if (m >= M) break;  // rows grow with rr: the rest are past M too
        const u32x4 v = ld16(stage + (rr + (lane >> 4)) * kQkvPitch + ch);
        float f[4] = {u2f(v[0]), u2f(v[1]), u2f(v[2]), u2f(v[3])};
        const bool rot = rope && t >= qa.prefix;  // the same for the row's 16 lanes
        float cs[4] = {0.0f, 0.0f, 0.0f, 0.0f}, sn[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (rot) {
            const int64_t trow = static_cast<int64_t>(t - qa.prefix) * 64 + ch;
            const float4 c4 = ld_f32x4(qa.cos_tab + trow), s4 = ld_f32x4(qa.sin_tab + trow);
            cs[0] = c4.x, cs[1] = c4.y, cs[2] = c4.z, cs[3] = c4.w;
            sn[0] = sg * s4.x, sn[1] = sg * s4.y, sn[2] = sg * s4.z, sn[3] = sg * s4.w;
        }
        if (norm)
            qk_norm_rope_vec<float, 16, true>(f, wr, br, qa.eps, rot, cs, sn);
        else
            qk_norm_rope_vec<float, 16, false>(f, wr, br, qa.eps, rot, cs, sn);
        u32x4 o;
        o[0] = f2u(f[0]), o[1] = f2u(f[1]), o[2] = f2u(f[2]), o[3] = f2u(f[3]);
        st16(obase + (static_cast<int64_t>(s) * qa.heads * qa.seq + t) * 64, o);
        m += 4;
        t += 4;
        while (t >= qa.seq) t -= qa.seq, s++;
    }
}

// The f32 tile kernel's epilogue, from a wave's accumulators (acc[a][b]
// register r of lane (l32, hh): column col0 + 32 a + 8 (r / 4) + 4 hh + r % 4, row
// row0 + 32 b + l32). For q|k|v every wave has left the main loop.
template <int EPI, int kRB>
__device__ __forceinline__ void f32_epilogue(const f32x16 (&acc)[2][kRB], float* smem, const float* bias,
                                             const float* gamma, const float* res, float* out, int64_t row0,
                                             int64_t col0, int M, int N, int wave, int lane, const QkvArgs& qa) {
    const int l32 = lane & 31, hh = lane >> 5;
    if constexpr (EPI == EPI_QKV) {
        // the stages' LDS takes the waves' blocks
        float* stage = smem + wave * (32 * kRB * kQkvPitch);
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++) {
                const int cl = 32 * a + 8 * r4 + 4 * hh;
                const float4 bv = bias ? ld_f32x4(bias + col0 + cl) : float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int b = 0; b < kRB; b++) {
                    u32x4 o;
                    o[0] = f2u(acc[a][b][4 * r4] + bv.x), o[1] = f2u(acc[a][b][4 * r4 + 1] + bv.y);
                    o[2] = f2u(acc[a][b][4 * r4 + 2] + bv.z), o[3] = f2u(acc[a][b][4 * r4 + 3] + bv.w);
                    st16(stage + (32 * b + l32) * kQkvPitch + cl, o);
                }
            }
        // only this wave reads its block back: a wave-level fence suffices
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        qkv_heads_out_f32(stage, qa, row0, M, col0, lane, 32 * kRB);
        return;
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) {
            const int64_t n = col0 + 32 * a + 8 * r4 + 4 * hh;
            const float4 bv = bias ? ld_f32x4(bias + n) : float4{0.0f, 0.0f, 0.0f, 0.0f};
            float4 gv = {0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (EPI == EPI_LS) gv = ld_f32x4(gamma + n);
#pragma unroll
            for (int b = 0; b < kRB; b++) {
                const int64_t m = row0 + 32 * b + l32;
                if (m >= M) continue;
                float v[4] = {acc[a][b][4 * r4] + bv.x, acc[a][b][4 * r4 + 1] + bv.y,
                              acc[a][b][4 * r4 + 2] + bv.z, acc[a][b][4 * r4 + 3] + bv.w};
                if constexpr (EPI == EPI_GELU) {
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = gelu_f(v[e]);
                }
                if constexpr (EPI == EPI_LS) {
                    // res + gamma * x, read and written by this lane only
                    // (res may be out)
                    const float4 rv = ld_f32x4(res + m * N + n);
                    v[0] = rv.x + gv.x * v[0], v[1] = rv.y + gv.y * v[1];
                    v[2] = rv.z + gv.z * v[2], v[3] = rv.w + gv.w * v[3];
                }
                u32x4 o;
                o[0] = f2u(v[0]), o[1] = f2u(v[1]), o[2] = f2u(v[2]), o[3] = f2u(v[3]);
                st16_nt(out + m * N + n, o);
            }
        }
}

// 4 floats normalised as hs_layernorm stores them.
__device__ __forceinline__ u32x4 ln_quad(u32x4 v, f32x2 st, float4 g, float4 b) {
    u32x4 o;
    o[0] = f2u(ln_affine(u2f(v[0]), st[0], st[1], g.x, b.x));
    o[1] = f2u(ln_affine(u2f(v[1]), st[0], st[1], g.y, b.y));
    o[2] = f2u(ln_affine(u2f(v[2]), st[0], st[1], g.z, b.z));
    o[3] = f2u(ln_affine(u2f(v[3]), st[0], st[1], g.w, b.w));
    return o;
}

// A wave's 32 kRB x 64 block of an f32 product on v_mfma_f32_32x32x2_f32,
// operands straight from memory (rows past M read row M - 1): MFMA j of a
// step takes element j of lane (l32, hh)'s 4 floats at 8 step + 4 hh of both rows.
template <bool LN, int kRB>
__device__ __forceinline__ void f32_block(f32x16 (&acc)[2][kRB], const float* x, const float* w, int64_t row0,
                                       int64_t col0, int M, int K, const LnArgs& la, int l32, int hh) {
    const float* xp[kRB];
    f32x2 st[kRB];
#pragma unroll
    for (int b = 0; b < kRB; b++) {
        const int64_t m = min(row0 + 32 * b + l32, static_cast<int64_t>(M) - 1);
        xp[b] = x + m * K + 4 * hh;
        if constexpr (LN) st[b] = *reinterpret_cast<const f32x2*>(la.stats + 2 * m);
    }
    const float* wp = w + (col0 + l32) * K + 4 * hh;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < kRB; b++) acc[a][b] = f32x16{};
#pragma unroll 1
    for (int k = 0; k < K; k += 8) {
        u32x4 av[2], bv[kRB];
#pragma unroll
        for (int a = 0; a < 2; a++) av[a] = ld16(wp + static_cast<int64_t>(32 * a) * K + k);
#pragma unroll
        for (int b = 0; b < kRB; b++) {
            bv[b] = ld16(xp[b] + k);
            if constexpr (LN)
                bv[b] = ln_quad(bv[b], st[b], ld_f32x4(la.ln_w + k + 4 * hh), ld_f32x4(la.ln_b + k + 4 * hh));
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int b = 0; b < kRB; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(u2f(av[a][j]), u2f(bv[b][j]), acc[a][b], 0, 0, 0);
    }
}

// ---------------------------------------------------------------------------
// f32 products on the bf16 matrix cores (N % 128 == 0, K % 32 == 0, the calls
// that few_rows does not give to gemm_skinny_kernel). The f32 matrix instructions run at a
// sixteenth of the bf16 rate; an f32 value is the sum of three bf16 ones
// (split3), a = h + m + l, and six products of those, every one exact in f32,
//     sum(h h)  +  sum(m m + m h + h m + l h + h l)
// give the f32 product to 2^-24 of each term, as one rounding of it would. The
// second sum, 2^-8 of the first, has accumulators of its own, so the chain of
// full-size roundings is K / 16 long instead of the f32 instructions' K / 2.
//
// The bf16 parts have f32's exponents, so this holds for every |a| from 2^-100
// up. An output whose x or w row has a smaller nonzero element, and one that
// comes out infinite or NaN, is computed again on v_mfma_f32_32x32x2_f32 (f32_block). That is decided
// for each output by its own two rows, so no result depends on what shares its
// tile.
//
// A workgroup of WM x WN waves computes 32 RB WM rows x 64 WN columns, a wave 32
// RB x 64 as out^T blocks. K goes in stages of 16 through LDS, two buffers of
// three planes (h, m, l) of 32-byte rows: chunk c (8 floats) of row r at c ^ ((r
// / 8) % 2), so sixteen rows' reads of a chunk and these writes cover the banks
// once. The f32 pieces are prefetched into registers and converted once per
// workgroup between the multiplies (7 vector instructions per element).
// Bounds: matrix issue (six MFMAs where f16 has one) with the conversion
// beside it. At 10992 rows, q|k|v / proj / fc1 / fc2, us: 390 / 140 / 500 / 486
// (165-190 TFLOP/s of f32 product) against 586 / 198 / 690 / 722 on the f32
// matrix cores; at 2748 rows 131 / 43 / 141 / 136 against 194 / 65 / 199 / 246.
// With two f16 parts and three products they were 273 / 100 / 346 / 312, but
// those parts keep no element below 2^-36 and only 22 bits of the others.
// Relative error against 64 bits, q|k|v and fc2: 1.9e-7 and 4.0e-7; the f32
// instructions 5.7e-7 and 1.15e-6. A 10992-row q|k|v with a row below 2^-100 in
// every tile, all computed twice: 1.05 ms. 256 x 128 and 128 x 256 tiles by 8
// waves: 478 and 471 us for q|k|v.
template <int WM, int WN, int RB_>
struct SplitTile {
    static constexpr int kWN = WN, kWaves = WM * WN, kThreads = 64 * kWaves, kRB = RB_;
    static constexpr int kBM = 32 * RB_ * WM, kBN = 64 * WN, kBK = 16;
    static constexpr int kPR = kThreads / 4;                                     // rows a pass of pieces covers
    static constexpr int kXP = kBM / kPR, kWP = kBN / kPR, kPieces = kXP + kWP;  // 4-float pieces per thread
    static_assert(kXP * kPR == kBM && kWP * kPR == kBN && kPR % 16 == 0, "pieces");
    struct Smem {
        uint16_t x[2][3][kBM * kBK];
        uint16_t w[2][3][kBN * kBK];
    };
    static constexpr size_t smem_bytes(int epi) {
        const size_t qkv = epi == EPI_QKV ? size_t{4} * kWaves * 32 * kRB * kQkvPitch : 0;
        return sizeof(Smem) > qkv ? sizeof(Smem) : qkv;
    }
};
using SplitShape = SplitTile<2, 2, 2>;   // 128 x 128, two workgroups per CU
using SplitEight = SplitTile<4, 2, 1>;   // 128 x 128 by 8 waves
using SplitNarrow = SplitTile<2, 2, 1>;  // 64 x 128
constexpr int kSplitKs = 32;             // K is a multiple: stages go in pairs

__device__ __forceinline__ u32x4 buf_ld16(__amdgpu_buffer_rsrc_t src, uint32_t voff, int soff) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src, voff, soff, 0));
}

template <int EPI, typename P, bool LN>
__global__ __launch_bounds__(P::kThreads, 2) void gemm_split_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    const float* __restrict__ gamma, const float* res, float* out, int M, int N, int K,
    int tiles_n, int ntiles, LnArgs la, QkvArgs qa) {
    constexpr int kRB = P::kRB, kXP = P::kXP, kPieces = P::kPieces;
    __shared__ __align__(16) unsigned char smem_raw[P::smem_bytes(EPI)];
    __shared__ uint8_t odd[P::kBM + P::kBN];  // x rows, then w rows, with an element below 2^-100
    __shared__ int any_odd;
    typename P::Smem& sm = *reinterpret_cast<typename P::Smem*>(smem_raw);
    const int tid = threadIdx.x;
    const int lane = lane_id(), wave = wave_in_block();
    const int l32 = lane & 31, hh = lane >> 5;
#if HS_GEMM_XCD
    // the f16 kernel's XCD-aware tile order
    const int per = static_cast<int>(gridDim.x / 8);
    const int tile = static_cast<int>(blockIdx.x % 8) * per + static_cast<int>(blockIdx.x / 8);
    if (tile >= ntiles) return;  // padding, before any barrier
#else
    const int tile = static_cast<int>(blockIdx.x);
#endif
    const int64_t m0 = static_cast<int64_t>(tile / tiles_n) * P::kBM;
    const int64_t n0 = static_cast<int64_t>(tile % tiles_n) * P::kBN;
    const int wm = (wave / P::kWN) * (32 * kRB);
    const int wn = (wave % P::kWN) * 64;
    for (int i = tid; i < P::kBM + P::kBN; i += P::kThreads) odd[i] = 0;
    if (tid == 0) any_odd = 0;

    const int xrows = static_cast<int>(min(static_cast<int64_t>(P::kBM), M - m0));
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(x + m0 * K), 0, xrows * K * 4, kRawBufferFlags);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(w + n0 * K), 0, P::kBN * K * 4, kRawBufferFlags);
    // Pieces 0 .. kXP of the thread are x's, the rest w's: piece i is row kPR i +
    // tid / 4 of its operand, floats 4 (tid % 4) .. + 4 of the stage (x rows
    // past M read row M - 1; their outputs are masked).
    const int prow = tid / 4, pc = tid % 4;
    uint32_t off[kPieces];
    f32x2 lst[kXP];
#pragma unroll
    for (int i = 0; i < kPieces; i++) {
        if (i < kXP) {
            const int row = static_cast<int>(min(m0 + P::kPR * i + prow, static_cast<int64_t>(M) - 1) - m0);
            off[i] = static_cast<uint32_t>(row * K * 4 + 16 * pc);
            if constexpr (LN) lst[i < kXP ? i : 0] = *reinterpret_cast<const f32x2*>(la.stats + 2 * (m0 + row));
        } else {
            off[i] = static_cast<uint32_t>((P::kPR * (i - kXP) + prow) * K * 4 + 16 * pc);
        }
    }
    // halves offset of a piece within its plane (kPR rows on: the same swizzle)
    const int dst = prow * 16 + 8 * ((pc >> 1) ^ ((prow >> 3) & 1)) + 4 * (pc & 1);

    // the next stage's pieces and the LayerNorm parameters of their columns
    u32x4 raw[kPieces];
    float4 lw, lb;
    SplitSmall small[kPieces];
    const int nsteps = K / P::kBK;  // even
    auto load_piece = [&](int i, int s) {
        raw[i] = buf_ld16(i < kXP ? xr : wr, off[i], s * 64);
        if constexpr (LN) {
            if (i == kXP - 1) {  // no x piece of the stage before needs them any more
                const int c = s * P::kBK + 4 * pc;
                lw = ld_f32x4(la.ln_w + c), lb = ld_f32x4(la.ln_b + c);
            }
        }
    };
    // Piece i into buffer buf, as h, m and l.
    auto store_piece = [&](int i, int buf) {
        u32x4 v = raw[i];
        if constexpr (LN) {
            if (i < kXP) v = ln_quad(v, lst[i < kXP ? i : 0], lw, lb);  // as hs_layernorm stores it
        }
        u32x2 part[3];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            uint32_t h, m, l;
            split3(u2f(v[2 * j]), u2f(v[2 * j + 1]), h, m, l);
            part[0][j] = h, part[1][j] = m, part[2][j] = l;
            small[i].note(u2f(v[2 * j]), u2f(v[2 * j + 1]));
        }
#pragma unroll
        for (int q = 0; q < 3; q++) {
            uint16_t* plane = i < kXP ? sm.x[buf][q] + P::kPR * 16 * i : sm.w[buf][q] + P::kPR * 16 * (i - kXP);
            *reinterpret_cast<u32x2*>(plane + dst) = part[q];
        }
    };

    // acc[a][b] (and the small products', acl): register r of lane (l32, hh) is
    // column wn + 32 a + 8 (r / 4) + 4 hh + r % 4, row wm + 32 b + l32
    f32x16 acc[2][kRB], acl[2][kRB];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < kRB; b++) acc[a][b] = f32x16{}, acl[a][b] = f32x16{};

    // operands: h of two stages, m and l of one
    u32x4 Ah[2][2], Bh[2][kRB], Am[2], Bm[kRB], Al[2], Bl[kRB];
    const int op = l32 * 16 + 8 * (hh ^ ((l32 >> 3) & 1));
    auto read_a = [&](u32x4(&d)[2], int q, int buf) {
#pragma unroll
        for (int a = 0; a < 2; a++) d[a] = ld16(sm.w[buf][q] + (wn + 32 * a) * 16 + op);
    };
    auto read_b = [&](u32x4(&d)[kRB], int q, int buf) {
#pragma unroll
        for (int b = 0; b < kRB; b++) d[b] = ld16(sm.x[buf][q] + (wm + 32 * b) * 16 + op);
    };
    auto multiply = [&](f32x16(&c)[2][kRB], const u32x4(&A)[2], const u32x4(&B)[kRB]) {
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < kRB; b++)
                c[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, A[a]),
                                                                 __builtin_bit_cast(bf16x8, B[b]), c[a][b], 0, 0, 0);
    };
#pragma unroll
    for (int i = 0; i < kPieces; i++) load_piece(i, 0);
#pragma unroll
    for (int i = 0; i < kPieces; i++) store_piece(i, 0);
#pragma unroll
    for (int i = 0; i < kPieces; i++) load_piece(i, 1);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // lgkmcnt(0) again, as an instruction the compiler knows: with scalar loads
    // pending, as far as it can tell, it would wait for every read of a stage
    // at the loop's top (395 us for q|k|v at 10992 rows against 390)
    __builtin_amdgcn_s_waitcnt(0xC07F);
    read_a(Ah[0], 0, 0);
    read_b(Bh[0], 0, 0);
    // A stage's six groups of multiplies. In the first four, stage s + 1 is
    // converted into the other buffer (last read before the barrier of the
    // stage before) and stage s + 2's pieces are loaded behind it; the barrier then opens stage s + 1, and its h operands are read under the
    // last group. cur = s % 2; NEXT: stage s + 1 exists.
    auto stage = [&](int s, auto cur_c, auto next_c) {
        constexpr bool NEXT = decltype(next_c)::value;
        constexpr int cur = decltype(cur_c)::value;
        const int ld = s + 2 < nsteps ? s + 2 : s + 1;  // (past the end: not used)
        auto convert = [&](int i) {
            if (NEXT && i < kPieces) {
                store_piece(i, cur ^ 1);
                load_piece(i, ld);
            }
        };
        // A group's reads, then its MFMAs with the conversion's vector work
        // between them; its loads leave with it (left to the compiler they
        // sink to the stage's end, a group before their use).
        auto group = [&](int reads, auto conv) {
            if (reads == 1) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // LDS reads
            if (reads == 2) __builtin_amdgcn_sched_group_barrier(0x100, 2 + kRB, 0);
#pragma unroll
            for (int q = 0; q < 2 * kRB; q++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // an MFMA
                if constexpr (NEXT && conv.value)
                    __builtin_amdgcn_sched_group_barrier(0x002, 16 / kRB, 0);  // VALU
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        constexpr std::true_type yes;
        constexpr std::false_type no;
        read_a(Am, 1, cur);
        read_b(Bm, 1, cur);
        convert(0);
        multiply(acc, Ah[cur], Bh[cur]);
        group(2, yes);
        convert(1);
        multiply(acl, Am, Bm);
        group(0, yes);
        convert(2);
        multiply(acl, Am, Bh[cur]);
        group(0, yes);
        read_a(Al, 2, cur);
        read_b(Bl, 2, cur);
        convert(3);
        multiply(acl, Ah[cur], Bm);
        group(2, yes);
        multiply(acl, Al, Bh[cur]);
        group(0, no);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if constexpr (NEXT) {
            read_a(Ah[cur ^ 1], 0, cur ^ 1);
            read_b(Bh[cur ^ 1], 0, cur ^ 1);
        }
        multiply(acl, Ah[cur], Bl);
        group(NEXT ? 2 : 0, no);
    };
    static_assert(kPieces <= 4, "one piece per group of multiplies");
    constexpr std::integral_constant<int, 0> even;
    constexpr std::integral_constant<int, 1> uneven;
    for (int s = 0; s + 2 < nsteps; s += 2) {
        stage(s, even, std::true_type{});
        stage(s + 1, uneven, std::true_type{});
    }
    stage(nsteps - 2, even, std::true_type{});
    stage(nsteps - 1, uneven, std::false_type{});

    // rows with an element below 2^-100 (a row's four threads are a quad)
#pragma unroll
    for (int i = 0; i < kPieces; i++) {
        if (small[i].seen()) {
            odd[(i < kXP ? P::kPR * i : P::kBM + P::kPR * (i - kXP)) + prow] = 1;
            any_odd = 1;
        }
    }
    __syncthreads();  // also: every wave has left the main loop
    float bad = 0.0f;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < kRB; b++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                acc[a][b][r] += acl[a][b][r];
                bad = fmaf(acc[a][b][r], 0.0f, bad);  // NaN once one is not finite
            }
    bool redo = !(bad == 0.0f);
    if (any_odd != 0)
        redo = redo || odd[P::kBM + wn + lane] != 0 || (lane < 32 * kRB && odd[wm + lane] != 0);
    if (__any(redo)) {
        f32x16 again[2][kRB];
        f32_block<LN, kRB>(again, x, w, m0 + wm, n0 + wn, M, K, la, l32, hh);
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < kRB; b++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const int row = wm + 32 * b + l32, col = wn + 32 * a + 8 * (r / 4) + 4 * hh + r % 4;
                    if (odd[row] != 0 || odd[P::kBM + col] != 0 || !(fabsf(acc[a][b][r]) <= 3.4028235e38f))
                        acc[a][b][r] = again[a][b][r];
                }
    }
    f32_epilogue<EPI, kRB>(acc, reinterpret_cast<float*>(smem_raw), bias, gamma, res, out, m0 + wm, n0 + wn, M, N, wave, lane, qa);
}

// ---------------------------------------------------------------------------
// few rows (f32, N % 128 == 0, K % 32 == 0, few_rows: up to 128):
// what such a call cannot do without is the weights' way from memory, so the
// work is split until every CU streams some of them. A workgroup of 16 waves
// takes 16 CB output columns x 16 RB rows; its waves share K, wave v taking
// the 128-byte pieces v, v + 16, .. of every row straight from memory into
// operand registers (16 rows x 128 bytes per pair of loads, no LDS stage, no
// barrier), and the 16 partial tiles are summed in wave order through LDS.
// v_mfma_f32_16x16x4_f32 computes out^T = w x^T: lane (r, g) holds row r's 4
// floats at chunk g of the piece's half and MFMA j takes element j of both
// operands; its accumulators are columns 4 g .. + 4 of output row r. The
// order of the sum depends on K only.
//
// At 8 rows (us, beside the tiles of gemm_split_kernel): 2048 x 2048 8.5 (55),
// 8192 x 2048 13.4 (53), 2048 x 8192 26 (200), i.e. 2.0-5.0 TB/s of weights; at
// 128 rows 18 (53), 64 (55), 64 (198); above, wide outputs are faster in tiles
// (200 rows, 8192 x 2048: 111 against 63).
constexpr int kSkinnyRows = 128;
constexpr int kSkWaves = 16, kSkThreads = 64 * kSkWaves;
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 sk_mfma(u32x4 a, u32x4 b, f32x4 c) {
#pragma unroll
    for (int j = 0; j < 4; j++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(u2f(a[j]), u2f(b[j]), c, 0, 0, 0);
    return c;
}

template <int EPI, int CB, int RB, bool LN>
__global__ __launch_bounds__(kSkThreads) void gemm_skinny_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    const float* __restrict__ gamma, const float* res, float* out, int M, int N, int K, int row_groups,
    int ngroups, QkvArgs qa, LnArgs la) {
    constexpr int kPiece = 32;                   // floats per 128 bytes
    constexpr int kTile = 256 * CB * RB;          // floats per partial tile
    constexpr int kStage = EPI == EPI_QKV ? 16 * RB * kQkvPitch : 0;
    static_assert(EPI != EPI_QKV || CB == 4, "a head is 64 columns");
    __shared__ __align__(16) float sm[kSkWaves * kTile + kStage];
    const int lane = lane_id(), wave = wave_in_block();
    const int r = lane & 15, g = lane >> 4;
    // an XCD takes a contiguous range, the row groups of one column group
    // (which share its weights) first; the grid is padded to 8
    const int per = static_cast<int>(gridDim.x / 8);
    const int grp = static_cast<int>(blockIdx.x % 8) * per + static_cast<int>(blockIdx.x / 8);
    if (grp >= ngroups) return;  // before any barrier
    const int64_t n0 = static_cast<int64_t>(grp / row_groups) * (16 * CB);
    const int64_t m0 = static_cast<int64_t>(grp % row_groups) * (16 * RB);

    const float* wp[CB];
    const float* xp[RB];
    f32x2 st[RB];
#pragma unroll
    for (int c = 0; c < CB; c++) wp[c] = w + (n0 + 16 * c + r) * K + g * 4;
#pragma unroll
    for (int b = 0; b < RB; b++) {
        // rows past M read row M - 1 (not stored)
        const int64_t m = min(m0 + 16 * b + r, static_cast<int64_t>(M) - 1);
        xp[b] = x + m * K + g * 4;
        if constexpr (LN) st[b] = *reinterpret_cast<const f32x2*>(la.stats + 2 * m);
    }
    f32x4 acc[CB][RB];
#pragma unroll
    for (int c = 0; c < CB; c++)
#pragma unroll
        for (int b = 0; b < RB; b++) acc[c][b] = f32x4{};
    u32x4 A[2][CB], B[2][RB];  // the piece's two halves
    auto load = [&](int k) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int c = 0; c < CB; c++) A[h][c] = ld16(wp[c] + k + 16 * h);
#pragma unroll
            for (int b = 0; b < RB; b++) B[h][b] = ld16(xp[b] + k + 16 * h);
        }
    };
    const int step = kSkWaves * kPiece;
    int k = wave * kPiece;
    if (k < K) load(k);
    while (k < K) {
        u32x4 a[2][CB], b[2][RB];
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int c = 0; c < CB; c++) a[h][c] = A[h][c];
#pragma unroll
            for (int i = 0; i < RB; i++) b[h][i] = B[h][i];
        }
        const int kc = k;
        k += step;
        if (k < K) load(k);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if constexpr (LN) {
#pragma unroll
                for (int i = 0; i < RB; i++) b[h][i] = ln_quad(b[h][i], st[i], ld_f32x4(la.ln_w + kc + 16 * h + 4 * g),
                                      ld_f32x4(la.ln_b + kc + 16 * h + 4 * g));
            }
#pragma unroll
            for (int c = 0; c < CB; c++)
#pragma unroll
                for (int i = 0; i < RB; i++) acc[c][i] = sk_mfma(a[h][c], b[h][i], acc[c][i]);
        }
    }
#pragma unroll
    for (int c = 0; c < CB; c++)
#pragma unroll
        for (int b = 0; b < RB; b++)
            *reinterpret_cast<f32x4*>(sm + wave * kTile + (c * RB + b) * 256 + r * 16 + 4 * g) = acc[c][b];
    __syncthreads();

    // quad q: columns 4 (q % 4) .. + 4 of row (q / 4) % 16 of block q / 64
    for (int q = threadIdx.x; q < kTile / 4; q += kSkThreads) {
        const int blk = q / 64, c = blk / RB, b = blk % RB;
        const int row = 16 * b + (q / 4) % 16, col = 16 * c + 4 * (q % 4);
        f32x4 v = *reinterpret_cast<const f32x4*>(sm + 4 * q);
#pragma unroll
        for (int i = 1; i < kSkWaves; i++) v += *reinterpret_cast<const f32x4*>(sm + i * kTile + 4 * q);
        const int64_t m = m0 + row, n = n0 + col;
        if (m >= M && EPI != EPI_QKV) continue;
        const float4 bv = bias ? ld_f32x4(bias + n) : float4{0.0f, 0.0f, 0.0f, 0.0f};
        float o[4] = {v[0] + bv.x, v[1] + bv.y, v[2] + bv.z, v[3] + bv.w};
        if constexpr (EPI == EPI_QKV) {
            // the head vectors' rows, staged behind the partial tiles
            *reinterpret_cast<float4*>(sm + kSkWaves * kTile + row * kQkvPitch + col) = float4{o[0], o[1], o[2], o[3]};
            continue;
        }
        if constexpr (EPI == EPI_GELU) {
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = gelu_f(o[e]);
        }
        if constexpr (EPI == EPI_LS) {
            // res + gamma * x (res may be out: each element is read and
            // written by one thread)
            const float4 gv = ld_f32x4(gamma + n), rv = ld_f32x4(res + m * N + n);
            o[0] = rv.x + gv.x * o[0], o[1] = rv.y + gv.y * o[1];
            o[2] = rv.z + gv.z * o[2], o[3] = rv.w + gv.w * o[3];
        }
        *reinterpret_cast<float4*>(out + m * N + n) = float4{o[0], o[1], o[2], o[3]};
    }
    if constexpr (EPI == EPI_QKV) {
        __syncthreads();
        // each wave takes 4 rows at a time in the row kernels' lane layout
        for (int r0 = 4 * wave; r0 < 16 * RB; r0 += 4 * kSkWaves)
            qkv_heads_out_f32(sm + kSkWaves * kTile + r0 * kQkvPitch, qa, m0 + r0, M, n0, lane, 4);
    }
}

// ---------------------------------------------------------------------------
// generic path: 64 x 64 output tile per 256 threads, 4 x 4 per thread,
// K in steps of 16 through LDS; f32 accumulation in K order.

constexpr int kGT = 64, kGK = 16;

template <typename T, int EPI, bool LN>
__global__ __launch_bounds__(256) void gemm_generic_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const float* __restrict__ bias,
    const float* __restrict__ gamma, const T* res, T* out, int M, int N, int K, int tiles_n,
    LnArgs la) {
    __shared__ float xs[kGK][kGT + 1];
    __shared__ float ws[kGK][kGT + 1];
    const int64_t m0 = static_cast<int64_t>(blockIdx.x / tiles_n) * kGT;
    const int64_t n0 = static_cast<int64_t>(blockIdx.x % tiles_n) * kGT;
    const int tr = threadIdx.x / 16, tc = threadIdx.x % 16;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += kGK) {
        for (int i = threadIdx.x; i < kGK * kGT; i += 256) {
            const int kk = i % kGK, rr = i / kGK;
            const int64_t xm = m0 + rr, wn = n0 + rr;
            const int kidx = k0 + kk;
            float xv = (xm < M && kidx < K) ? static_cast<float>(x[xm * K + kidx]) : 0.0f;
            if constexpr (LN) {
                // the element as hs_layernorm stores it
                if (xm < M && kidx < K)
                    xv = storage_round(ln_affine(xv, la.stats[2 * xm], la.stats[2 * xm + 1],
                                                 la.ln_w[kidx], la.ln_b[kidx]),
                                       T{});
            }
            xs[kk][rr] = xv;
            ws[kk][rr] = (wn < N && kidx < K) ? static_cast<float>(w[wn * K + kidx]) : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kGK; kk++) {
            float xv[4], wv[4];
#pragma unroll
            for (int i = 0; i < 4; i++) xv[i] = xs[kk][tr * 4 + i], wv[i] = ws[kk][tc * 4 + i];
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] += xv[i] * wv[j];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int64_t m = m0 + tr * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t n = n0 + tc * 4 + j;
            if (n >= N) continue;
            float v = acc[i][j] + (bias ? bias[n] : 0.0f);
            if constexpr (EPI == EPI_GELU) v = gelu_f(v);
            if constexpr (EPI == EPI_LS)
                v = static_cast<float>(res[m * N + n]) + gamma[n] * storage_round(v, T{});
            out[m * N + n] = static_cast<T>(v);
        }
    }
}

bool fast_shape(hs_dtype dt, int N, int K, const void* x, const void* w, const float* bias,
                const float* gamma, const void* out, const void* res) {
    // K == 0 takes the generic kernel (out = bias): the fast path's first
    // stage would read K-tiles that do not exist
    // K <= 2^20 keeps a tile's byte offsets (256 rows x K x 2) in 32 bits
    return dt == HS_F16 && N % F16Big::kBN == 0 && K > 0 && K % kBK == 0 && K <= (1 << 20) && aligned16(x) && aligned16(w) &&
           (!bias || aligned16(bias)) && (!gamma || aligned16(gamma)) && aligned16(out) &&
           (!res || aligned16(res));
}

// Fast-path eligibility of a call, decided before anything is enqueued.
template <bool LN>
bool takes_fast_path(hs_dtype dt, int N, int K, const void* x, const void* w, const float* bias,
                     const float* gamma, const void* out, const void* res, const LnArgs& la) {
    return fast_shape(dt, N, K, x, w, bias, gamma, out, res) &&
           (!LN || (aligned16(la.ln_w) && aligned16(la.ln_b)));
}

constexpr int kF32ColTile = 128;  // columns of an f32 tile: N is a multiple of it

// f32 matrix-core eligibility: shape and alignment.
bool f32_fast(hs_dtype dt, int N, int K, const void* x, const void* w, const float* bias,
              const float* gamma, const void* out, const void* res) {
    // K <= 2^19 keeps a tile's byte offsets (128 rows x K x 4) in 32 bits
    return dt == HS_F32 && N % kF32ColTile == 0 && K > 0 && K % kSplitKs == 0 &&
           K <= (1 << 19) && aligned16(x) && aligned16(w) && (!bias || aligned16(bias)) &&
           (!gamma || aligned16(gamma)) && aligned16(out) && (!res || aligned16(res));
}

template <int EPI, typename P, bool LN>
void launch_split_as(hipStream_t st, const void* x, const void* w, const float* bias, const float* gamma,
                     const void* res, void* out, int M, int N, int K, const LnArgs& la, const QkvArgs& qa) {
    const int tiles_n = N / P::kBN;
    const int64_t ntiles = ceil_div(M, P::kBM) * tiles_n;
    const int64_t blocks = HS_GEMM_XCD ? ceil_div(ntiles, 8) * 8 : ntiles;
    gemm_split_kernel<EPI, P, LN><<<dim3(static_cast<uint32_t>(blocks)), dim3(P::kThreads), 0, st>>>(
        static_cast<const float*>(x), static_cast<const float*>(w), bias, gamma,
        static_cast<const float*>(res), static_cast<float*>(out), M, N, K, tiles_n,
        static_cast<int>(ntiles), la, qa);
}

// 128 x 128 tiles by two 4-wave workgroups per CU; where one per CU holds
// them all, by one of 8 waves (2748 rows, fc2: 135 us against 152), and where half
// the CUs would, in 64 x 128 tiles (1374 rows, fc2: 111 us against 148 and 123).
// Every shape sums k in one order, and computes the same outputs again.
template <int EPI, bool LN>
void launch_split(hipStream_t st, const void* x, const void* w, const float* bias, const float* gamma,
                  const void* res, void* out, int M, int N, int K, const LnArgs& la, const QkvArgs& qa) {
    const int64_t tiles = ceil_div(M, SplitShape::kBM) * (N / SplitShape::kBN), cus = num_cus();
    if (2 * tiles <= cus)
        launch_split_as<EPI, SplitNarrow, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
    else if (tiles <= cus)
        launch_split_as<EPI, SplitEight, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
    else
        launch_split_as<EPI, SplitShape, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
}

// Whether the few-row kernel takes a call: by its shape alone, and so that a
// product summed in parts of its columns, as q, k and v apart, takes one route
// with the whole where the whole is promised their bits (8, 16 or 32 heads, i.e.
// up to 6144 columns). Wide outputs of more than 32 rows make too many
// workgroups, each reading its weights again: 1024 deep, us here and in tiles:
// 128 rows, 6144 columns 27, 30; 8192 35, 30; 16384 72, 36; 64 rows, 32768
// columns 70, 48; 32 rows, 32768 columns 36, 43; q|k|v of 128 rows and 32 heads
// 35, 34; 64 heads 68, 34.
template <int EPI>
bool few_rows(int M, int N) {
    if (M > kSkinnyRows) return false;
    if constexpr (EPI == EPI_QKV)
        return N <= 6144 || N / 64 * ceil_div(M, 16) <= 512;
    else
        return N <= 2048 || M <= 32 || N * ceil_div(M, 32) <= 24576;
}

template <int EPI, int CB, int RB, bool LN>
void launch_skinny_as(hipStream_t st, const float* x, const float* w, const float* bias, const float* gamma,
                      const float* res, float* out, int M, int N, int K, const LnArgs& la, const QkvArgs& qa) {
    const int row_groups = static_cast<int>(ceil_div(M, 16 * RB));
    const int ngroups = N / (16 * CB) * row_groups;
    const int64_t blocks = ceil_div(ngroups, 8) * 8;
    gemm_skinny_kernel<EPI, CB, RB, LN><<<dim3(static_cast<uint32_t>(blocks)), dim3(kSkThreads), 0, st>>>(
        x, w, bias, gamma, res, out, M, N, K, row_groups, ngroups, qa, la);
}

// The smallest tile whose workgroups the CUs hold at once (8 rows: 2048
// columns 1 x 1 8.4 us, 2 x 1 11.9; 8192 columns 16.4, 14.2; 33 rows of 6144: 2 x 2
// 32.9, 2 x 3 23.3), and 2 x 2 where none does (100 rows of 8192: 2 x 1 82, 2
// x 2 65, 2 x 3 67).
template <int EPI, bool LN>
void launch_skinny(hipStream_t st, const void* x_, const void* w_, const float* bias, const float* gamma,
                   const void* res_, void* out_, int M, int N, int K, const LnArgs& la, const QkvArgs& qa) {
    const float *x = static_cast<const float*>(x_), *w = static_cast<const float*>(w_);
    const float* res = static_cast<const float*>(res_);
    float* out = static_cast<float*>(out_);
    if constexpr (EPI == EPI_QKV) {
        launch_skinny_as<EPI, 4, 1, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
    } else {
        const int64_t cus = num_cus();
        auto groups = [&](int cb, int rb) { return N / (16 * cb) * ceil_div(M, 16 * rb); };
        if (groups(1, 1) <= cus)
            launch_skinny_as<EPI, 1, 1, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
        else if (groups(2, 1) <= cus)
            launch_skinny_as<EPI, 2, 1, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
        else if (groups(2, 2) > cus && groups(2, 3) <= cus)
            launch_skinny_as<EPI, 2, 3, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
        else
            launch_skinny_as<EPI, 2, 2, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
    }
}

template <int EPI, typename P, bool LN>
void launch_f16(hipStream_t st, const void* x, const void* w, const float* bias, const float* gamma,
                const void* res, void* out, int M, int N, int K, const LnArgs& la, const QkvArgs& qa) {
    const int tiles_n = N / P::kBN;
    const int64_t ntiles = ceil_div(M, P::kBM) * tiles_n;
    const int64_t blocks = HS_GEMM_XCD ? ceil_div(ntiles, 8) * 8 : ntiles;
    gemm_f16_kernel<EPI, P, LN><<<dim3(static_cast<uint32_t>(blocks)), dim3(P::kThreads), 0, st>>>(
        static_cast<const f16*>(x), static_cast<const f16*>(w), bias, gamma,
        static_cast<const f16*>(res), static_cast<f16*>(out), M, N, K, tiles_n,
        static_cast<int>(ntiles), qa, la);
}

template <int EPI, bool LN = false>
hs_status launch(hipStream_t st, hs_dtype dt, const void* x, const void* w, const float* bias,
                 const float* gamma, const void* res, void* out, int M, int N, int K,
                 const char* op, const QkvArgs& qa = QkvArgs{}, const LnArgs& la = LnArgs{}) {
    if (f32_fast(dt, N, K, x, w, bias, gamma, out, res) &&
        (!LN || (aligned16(la.ln_w) && aligned16(la.ln_b)))) {
        if (few_rows<EPI>(M, N))
            launch_skinny<EPI, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
        else
            launch_split<EPI, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
        return check_launch(op);
    }
    if (takes_fast_path<LN>(dt, N, K, x, w, bias, gamma, out, res, la)) {
        // The tile shape. Every shape sums k in the same order, so the choice
        // changes no bit of the result (the LayerNorm prologue exists for
        // F16Big). Times in us for the q|k|v / proj / fc1 / fc2 shapes, Small
        // / Solo / Pair / Mid / Big:
        //   64 x 64 while two per CU hold them all (S=1, 1386 rows: proj
        //     8.6 / 10 / 11 / 20 / 24, fc2 23 / 28 / 43 / 66 / 78);
        //   then 128 x 128 with four stages while one per CU does (S=2: proj
        //     16 / 11.4 / 12.7 / 21 / 26, fc2 49 / 31 / 44 / 66 / 78), or
        //     with two stages while two per CU do (S=4 proj 27 / 24 / 20 / 24
        //     / 29, S=1 q|k|v 25 / 22 / 16 / 21 / 24);
        //   beyond, the fewer rounds of the chip in rows, with a tenth on Mid
        //     for its larger share of LDS reads (S=2 q|k|v - / 36 / 31 / 23 /
        //     26, S=8 q|k|v Mid 76, Big 87; fc1 at 11088 rows 119, 111).
        if constexpr (LN) {
            launch_f16<EPI, F16Big, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
        } else {
            const int64_t cus = num_cus();
            auto tiles = [&](int bm, int bn) { return ceil_div(M, bm) * (N / bn); };
            const int64_t t128 = tiles(128, 128);
            if (tiles(64, 64) <= 2 * cus)
                launch_f16<EPI, F16Small, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
            else if (t128 <= cus)
                launch_f16<EPI, F16Solo, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
            else if (t128 <= 2 * cus)
                launch_f16<EPI, F16Pair, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
            else if (ceil_div(tiles(192, 256), cus) * 192 * 11 < ceil_div(tiles(256, 256), cus) * 256 * 10)
                launch_f16<EPI, F16Mid, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
            else
                launch_f16<EPI, F16Big, LN>(st, x, w, bias, gamma, res, out, M, N, K, la, qa);
        }
        return check_launch(op);
    }
    if constexpr (EPI == EPI_QKV) {
        return fail(HS_EUNSUPPORTED,
                    "%s: needs K %% %d == 0 (f16) or %% %d == 0 (f32) and 16-byte aligned buffers", op,
                    kBK, kSplitKs);
    } else {
        const int tiles_n = static_cast<int>(ceil_div(N, kGT));
        const int64_t blocks = ceil_div(M, kGT) * tiles_n;
        if (dt == HS_F16)
            gemm_generic_kernel<f16, EPI, LN><<<dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, st>>>(
                static_cast<const f16*>(x), static_cast<const f16*>(w), bias, gamma,
                static_cast<const f16*>(res), static_cast<f16*>(out), M, N, K, tiles_n, la);
        else
            gemm_generic_kernel<float, EPI, LN><<<dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, st>>>(
                static_cast<const float*>(x), static_cast<const float*>(w), bias, gamma,
                static_cast<const float*>(res), static_cast<float*>(out), M, N, K, tiles_n, la);
        return check_launch(op);
    }
}

hs_status check(const char* op, hs_dtype dt, const void* x, const void* w, const void* res,
                const void* out, int64_t M, int32_t N, int32_t K, bool needs_res) {
    if (!valid_dtype(dt)) return fail(HS_EINVAL, "%s: unknown dtype", op);
    if (M < 0 || N < 0 || K < 0) return fail(HS_EINVAL, "%s: shape M=%lld N=%d K=%d", op, static_cast<long long>(M), N, K);
    if (M >= (int64_t{1} << 31) || M * N >= (int64_t{1} << 40) || M * K >= (int64_t{1} << 40))
        return fail(HS_EINVAL, "%s: too large", op);
    if (M == 0 || N == 0) return HS_OK;
    if (!x || !w || !out || (needs_res && !res)) return fail(HS_EINVAL, "%s: null buffer", op);
    const int64_t esz = dtype_size(dt);
    const int64_t ob = M * N * esz;
    if (overlaps(out, ob, x, M * K * esz) || overlaps(out, ob, w, int64_t{N} * K * esz))
        return fail(HS_EINVAL, "%s: out overlaps x or w", op);
    if (needs_res && res != out && overlaps(out, ob, res, ob))
        return fail(HS_EINVAL, "%s: out partially overlaps res", op);
    return HS_OK;
}

}  // namespace
}  // namespace hs

extern "C" hs_status hs_linear(hs_stream_t stream, hs_dtype dt, const void* x, const void* w,
                               const float* bias, void* out, int64_t m, int32_t n, int32_t k) {
    using namespace hs;
    const hs_status rc = check("linear", dt, x, w, nullptr, out, m, n, k, false);
    if (rc != HS_OK || m == 0 || n == 0) return rc;
    return launch<EPI_BIAS>(static_cast<hipStream_t>(stream), dt, x, w, bias, nullptr, nullptr, out,
                            static_cast<int>(m), n, k, "linear");
}

extern "C" hs_status hs_linear_gelu(hs_stream_t stream, hs_dtype dt, const void* x, const void* w,
                                    const float* bias, void* out, int64_t m, int32_t n, int32_t k) {
    using namespace hs;
    const hs_status rc = check("linear_gelu", dt, x, w, nullptr, out, m, n, k, false);
    if (rc != HS_OK || m == 0 || n == 0) return rc;
    return launch<EPI_GELU>(static_cast<hipStream_t>(stream), dt, x, w, bias, nullptr, nullptr, out,
                            static_cast<int>(m), n, k, "linear_gelu");
}

extern "C" hs_status hs_linear_ls_residual(hs_stream_t stream, hs_dtype dt, const void* x,
                                           const void* w, const float* bias, const float* gamma,
                                           const void* res, void* out, int64_t m, int32_t n,
                                           int32_t k) {
    using namespace hs;
    if (!gamma && m > 0 && n > 0) return fail(HS_EINVAL, "linear_ls_residual: null gamma");
    const hs_status rc = check("linear_ls_residual", dt, x, w, res, out, m, n, k, true);
    if (rc != HS_OK || m == 0 || n == 0) return rc;
    return launch<EPI_LS>(static_cast<hipStream_t>(stream), dt, x, w, bias, gamma, res, out,
                          static_cast<int>(m), n, k, "linear_ls_residual");
}

namespace hs {
namespace {

// Validation and arguments of the q|k|v projection with heads (shared by
// hs_linear_qkv_heads and hs_linear_ln_qkv_heads). Returns HS_OK with
// *skip set for zero-size work.
hs_status qkv_setup(const char* op, hs_dtype dt, const void* x, const void* w_qkv,
                    const float* qn_w, const float* qn_b, const float* kn_w, const float* kn_b,
                    const float* sin_tab, const float* cos_tab, void* q_out, void* k_out,
                    void* v_out, int32_t S, int32_t T, int32_t H, int32_t d, int32_t k,
                    int32_t prefix, float eps, QkvArgs* qa, bool* skip) {
    *skip = false;
    if (!valid_dtype(dt)) return fail(HS_EINVAL, "%s: unknown dtype", op);
    if (S < 0 || T < 0 || H <= 0 || d <= 0 || k <= 0)
        return fail(HS_EINVAL, "%s: shape S=%d T=%d H=%d d=%d k=%d", op, S, T, H, d, k);
    if (prefix < 0 || prefix > T) return fail(HS_EINVAL, "%s: prefix %d outside [0, %d]", op, prefix, T);
    if ((qn_w == nullptr) != (qn_b == nullptr) || (kn_w == nullptr) != (kn_b == nullptr))
        return fail(HS_EINVAL, "%s: a norm needs both weight and bias", op);
    if ((sin_tab == nullptr) != (cos_tab == nullptr))
        return fail(HS_EINVAL, "%s: RoPE needs both tables", op);
    if (!(eps > 0.0f)) return fail(HS_EINVAL, "%s: eps must be positive", op);
    const int64_t M = int64_t{S} * T;
    const int64_t N = int64_t{3} * H * d;
    if (N >= (int64_t{1} << 31) || M >= (int64_t{1} << 31) || M * N >= (int64_t{1} << 40) ||
        M * k >= (int64_t{1} << 40))
        return fail(HS_EINVAL, "%s: too large", op);
    if (M == 0) {
        *skip = true;
        return HS_OK;
    }
    if (!x || !w_qkv || !q_out || !k_out || !v_out) return fail(HS_EINVAL, "%s: null buffer", op);
    const int64_t esz = dtype_size(dt), ob = M * H * d * esz;  // each of q, k, v
    const void* outs[3] = {q_out, k_out, v_out};
    for (int i = 0; i < 3; i++) {
        if (overlaps(outs[i], ob, x, M * k * esz) || overlaps(outs[i], ob, w_qkv, N * k * esz))
            return fail(HS_EINVAL, "%s: an output overlaps x or w", op);
        for (int j = 0; j < i; j++)
            if (overlaps(outs[i], ob, outs[j], ob)) return fail(HS_EINVAL, "%s: outputs overlap", op);
    }
    // The fused epilogue needs one head per wave (64 columns) and whole
    // column tiles (256 in f16, 128 in f32); other shapes run linear then
    // qknorm_rope.
    const int64_t tile_n = dt == HS_F16 ? F16Big::kBN : kF32ColTile;
    if (d != 64 || N % tile_n != 0)
        return fail(HS_EUNSUPPORTED, "%s: needs head dim 64 and 3*H*64 %% %lld == 0", op,
                    static_cast<long long>(tile_n));
    const float* params[6] = {qn_w, qn_b, kn_w, kn_b, sin_tab, cos_tab};
    for (const float* p : params)
        if (p && !aligned16(p)) return fail(HS_EUNSUPPORTED, "%s: parameters must be 16-byte aligned", op);
    if (!aligned16(k_out) || !aligned16(v_out))
        return fail(HS_EUNSUPPORTED, "%s: outputs must be 16-byte aligned", op);
    *qa = QkvArgs{};
    qa->out[0] = q_out, qa->out[1] = k_out, qa->out[2] = v_out;
    qa->nw[0] = qn_w, qa->nb[0] = qn_b, qa->nw[1] = kn_w, qa->nb[1] = kn_b;
    qa->sin_tab = sin_tab, qa->cos_tab = cos_tab;
    qa->seq = T, qa->heads = H, qa->prefix = prefix, qa->eps = eps;
    return HS_OK;
}

// A byte range that the LayerNorm prologue's workspace must not overlap.
struct Span {
    const void* p;
    int64_t bytes;
};

// Checks of the LayerNorm prologue's operands: ln_w and ln_b (k f32 each)
// and the workspace (2 m floats, 8-byte aligned), which receives each x
// row's (mean, rstd) and so must not overlap any buffer the call reads or
// writes (`spans`).
hs_status ln_check(const char* op, const float* ln_w, const float* ln_b, const float* workspace,
                   int64_t M, int32_t K, float eps, std::initializer_list<Span> spans) {
    if (!ln_w || !ln_b || !workspace) return fail(HS_EINVAL, "%s: null buffer", op);
    if (!(eps > 0.0f)) return fail(HS_EINVAL, "%s: eps must be positive", op);
    if (reinterpret_cast<uintptr_t>(workspace) % 8 != 0)
        return fail(HS_EINVAL, "%s: workspace must be 8-byte aligned", op);
    const int64_t wsb = M * 8;
    if (overlaps(workspace, wsb, ln_w, int64_t{K} * 4) ||
        overlaps(workspace, wsb, ln_b, int64_t{K} * 4))
        return fail(HS_EINVAL, "%s: workspace overlaps the LayerNorm parameters", op);
    for (const Span& sp : spans)
        if (sp.p && overlaps(workspace, wsb, sp.p, sp.bytes))
            return fail(HS_EINVAL, "%s: workspace overlaps an operand", op);
    return HS_OK;
}

// hs_linear_ln / hs_linear_ln_gelu (and the allocation-free variant): the
// row statistics into ws, then the product with the LayerNorm prologue.
template <int EPI>
hs_status linear_ln_entry(const char* op, hipStream_t st, hs_dtype dt, const void* x,
                          const float* ln_w, const float* ln_b, const void* w, const float* bias,
                          float* ws, void* out, int64_t m, int32_t n, int32_t k, float eps) {
    hs_status rc = check(op, dt, x, w, nullptr, out, m, n, k, false);
    if (rc != HS_OK || m == 0 || n == 0) return rc;
    if (k == 0) return fail(HS_EINVAL, "%s: k must be positive", op);
    const int64_t esz = dtype_size(dt);
    rc = ln_check(op, ln_w, ln_b, ws, m, k, eps,
                  {{x, m * k * esz}, {w, int64_t{n} * k * esz}, {bias, int64_t{n} * 4},
                   {out, m * n * esz}});
    if (rc != HS_OK) return rc;
    // (a failure keeps the statistics launch's own message)
    rc = hs_layernorm_stats(st, dt, x, ws, m, k, eps);
    if (rc != HS_OK) return rc;
    return launch<EPI, true>(st, dt, x, w, bias, nullptr, nullptr, out, static_cast<int>(m), n, k,
                             op, QkvArgs{}, LnArgs{ws, ln_w, ln_b});
}

}  // namespace
}  // namespace hs

extern "C" hs_status hs_linear_qkv_heads(hs_stream_t stream, hs_dtype dt, const void* x,
                                         const void* w_qkv, const float* b_qkv, const float* qn_w,
                                         const float* qn_b, const float* kn_w, const float* kn_b,
                                         const float* sin_tab, const float* cos_tab, void* q_out,
                                         void* k_out, void* v_out, int32_t S, int32_t T,
                                         int32_t H, int32_t d, int32_t k, int32_t prefix,
                                         float eps) {
    using namespace hs;
    const char* op = "linear_qkv_heads";
    QkvArgs qa;
    bool skip;
    const hs_status rc = qkv_setup(op, dt, x, w_qkv, qn_w, qn_b, kn_w, kn_b, sin_tab, cos_tab,
                                   q_out, k_out, v_out, S, T, H, d, k, prefix, eps, &qa, &skip);
    if (rc != HS_OK || skip) return rc;
    const int64_t M = int64_t{S} * T, N = int64_t{3} * H * d;
    return launch<EPI_QKV>(static_cast<hipStream_t>(stream), dt, x, w_qkv, b_qkv, nullptr, nullptr,
                           q_out, static_cast<int>(M), static_cast<int>(N), k, op, qa);
}

extern "C" hs_status hs_linear_ln(hs_stream_t stream, hs_dtype dt, const void* x,
                                  const float* ln_w, const float* ln_b, const void* w,
                                  const float* bias, float* workspace, void* out, int64_t m,
                                  int32_t n, int32_t k, float eps) {
    return hs::linear_ln_entry<hs::EPI_BIAS>("linear_ln", static_cast<hipStream_t>(stream), dt, x,
                                             ln_w, ln_b, w, bias, workspace, out, m, n, k, eps);
}

extern "C" hs_status hs_linear_ln_gelu(hs_stream_t stream, hs_dtype dt, const void* x,
                                       const float* ln_w, const float* ln_b, const void* w,
                                       const float* bias, float* workspace, void* out, int64_t m,
                                       int32_t n, int32_t k, float eps) {
    return hs::linear_ln_entry<hs::EPI_GELU>("linear_ln_gelu", static_cast<hipStream_t>(stream), dt,
                                             x, ln_w, ln_b, w, bias, workspace, out, m, n, k, eps);
}

extern "C" hs_status hs_linear_ln_qkv_heads(hs_stream_t stream, hs_dtype dt, const void* x,
                                            const float* ln_w, const float* ln_b,
                                            const void* w_qkv, const float* b_qkv,
                                            const float* qn_w, const float* qn_b,
                                            const float* kn_w, const float* kn_b,
                                            const float* sin_tab, const float* cos_tab,
                                            float* workspace, void* q_out, void* k_out,
                                            void* v_out, int32_t S, int32_t T, int32_t H,
                                            int32_t d, int32_t k, int32_t prefix, float eps) {
    using namespace hs;
    const char* op = "linear_ln_qkv_heads";
    QkvArgs qa;
    bool skip;
    hs_status rc = qkv_setup(op, dt, x, w_qkv, qn_w, qn_b, kn_w, kn_b, sin_tab, cos_tab, q_out,
                             k_out, v_out, S, T, H, d, k, prefix, eps, &qa, &skip);
    if (rc != HS_OK || skip) return rc;
    const int64_t M = int64_t{S} * T, N = int64_t{3} * H * d;
    const int64_t esz = dtype_size(dt), ob = M * H * d * esz;
    const int64_t tab = int64_t{T - prefix} * d * 4;
    rc = ln_check(op, ln_w, ln_b, workspace, M, k, eps,
                  {{x, M * k * esz}, {w_qkv, N * k * esz}, {b_qkv, N * 4}, {qn_w, d * 4},
                   {qn_b, d * 4}, {kn_w, d * 4}, {kn_b, d * 4}, {sin_tab, tab}, {cos_tab, tab},
                   {q_out, ob}, {k_out, ob}, {v_out, ob}});
    if (rc != HS_OK) return rc;
    const LnArgs la{workspace, ln_w, ln_b};
    // the q|k|v epilogue exists on the matrix-core path only: refuse other
    // calls before the statistics are enqueued
    const bool f32_ok = f32_fast(dt, static_cast<int>(N), k, x, w_qkv, b_qkv, nullptr, q_out, nullptr) &&
                        aligned16(ln_w) && aligned16(ln_b);
    if (!f32_ok && !takes_fast_path<true>(dt, static_cast<int>(N), k, x, w_qkv, b_qkv, nullptr, q_out,
                                          nullptr, la))
        return fail(HS_EUNSUPPORTED,
                    "%s: needs K %% %d == 0 (f16) or %% %d == 0 (f32) and 16-byte aligned buffers", op,
                    kBK, kSplitKs);
    hipStream_t st = static_cast<hipStream_t>(stream);
    rc = hs_layernorm_stats(st, dt, x, workspace, M, k, eps);
    if (rc != HS_OK) return rc;
    return launch<EPI_QKV, true>(st, dt, x, w_qkv, b_qkv, nullptr, nullptr, q_out,
                                 static_cast<int>(M), static_cast<int>(N), k, op, qa, la);
}

// ---------------------------------------------------------------------------
// An allocation-free variant of hs_linear_ln_gelu: the row statistics live
// in a file-scope device array instead of a caller workspace. Each device the
// library runs on holds its own copy for the life of the process; its device
// address comes from hipGetSymbolAddress, taken once per device (with that
// device current) on the first call there. Every call on a device shares
// that device's array, so calls that overlap on one device race; the array
// keeps the last call's statistics, and each call writes every row it reads.

namespace hs {
namespace {

constexpr int64_t kNoAllocMaxRows = int64_t{1} << 19;  // 524,288 rows: 4 MiB of statistics
static __device__ __align__(256) float scratch[2 * kNoAllocMaxRows];

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch[kScratchDevices];  // device address of `scratch` per device, once taken

// The current device's address of `scratch` (nullptr with *rc and the
// error message set on failure). The array's host-side name is not a device
// address: only the pointer returned by hipGetSymbolAddress goes to kernels.
float* scratch_address(const char* op, hs_status* rc) {
    int dev = 0;
    const hipError_t de = hipGetDevice(&dev);
    if (de != hipSuccess) {
        *rc = fail(HS_EHIP, "%s: hipGetDevice: %s", op, hipGetErrorString(de));
        return nullptr;
    }
    if (dev < 0 || dev >= kScratchDevices) {
        *rc = fail(HS_EUNSUPPORTED, "%s: device %d beyond the %d the library tracks", op, dev,
                   kScratchDevices);
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch[dev] == nullptr) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || ptr == nullptr) {
            *rc = fail(HS_EHIP, "%s: hipGetSymbolAddress(scratch): %s", op, hipGetErrorString(e));
            return nullptr;
        }
        g_scratch[dev] = static_cast<float*>(ptr);
    }
    return g_scratch[dev];
}

}  // namespace
}  // namespace hs

extern "C" hs_status hs_linear_ln_gelu_noalloc(hs_stream_t stream, hs_dtype dt, const void* x,
                                               const float* ln_w, const float* ln_b,
                                               const void* w, const float* bias, void* out,
                                               int64_t m, int32_t n, int32_t k, float eps) {
    using namespace hs;
    const char* op = "linear_ln_gelu_noalloc";
    if (m > kNoAllocMaxRows)
        return fail(HS_EINVAL, "%s: m = %lld rows exceeds the statistics array's %lld", op,
                    static_cast<long long>(m), static_cast<long long>(kNoAllocMaxRows));
    if (m <= 0 || n <= 0)  // the shape checks and zero-size returns of the workspace entry
        return linear_ln_entry<EPI_GELU>(op, static_cast<hipStream_t>(stream), dt, x, ln_w, ln_b,
                                         w, bias, nullptr, out, m, n, k, eps);
    hs_status rc = HS_OK;
    float* ws = scratch_address(op, &rc);
    if (ws == nullptr) return rc;
    return linear_ln_entry<EPI_GELU>(op, static_cast<hipStream_t>(stream), dt, x, ln_w, ln_b, w,
                                     bias, ws, out, m, n, k, eps);
}
