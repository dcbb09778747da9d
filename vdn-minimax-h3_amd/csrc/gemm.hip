// fp8 x fp8 GEMM with per-token x per-output-channel dequantization and a
// fused bias / GELU(tanh) / AdaLN-gate epilogue, for gfx950 (MI355X).
//
//   v         = bf16(x_scale[m] * w_scale[n] * sum_k xq[m][k] wq[n][k])
//   v         = bf16(v + bias[n])                          (with a bias)
//   out[m][n] = bf16(epi(v))                               (none / GELU(tanh) / gate)
// rounding to bf16 where the reference's op sequence does (_scaled_mm with
// out_dtype=bf16, the bf16 bias add, then the epilogue on the bf16 tensor).
//
// Both operands are K-contiguous (xq [M, K], wq [N, K]), the "TN" layout of
// torch._scaled_mm(x_fp8, weight_fp8.t()) in the reference (fp8_linear.py:272).
//
// Main kernel (K % 256 == 0). A workgroup of 4 wavefronts computes a 256 (m) x
// 256 (n) output tile; each wave owns a 128 x 128 quadrant as 8 x 8
// v_mfma_f32_16x16x128_f8f6f4 tiles (256 fp32 accumulators per lane, in AGPRs).
// K advances in 128-byte blocks through two LDS stages (X and W tiles of 256
// rows x 128 bytes: 64 KiB a stage). Global -> LDS copies bypass VGPRs
// (buffer_load_dwordx4 ... lds) and move whole 128-byte rows -- half-line
// copies stream at two thirds of the rate on this part. A block is 64 MFMAs,
// each over the whole 128 K bytes: 8 groups, group j multiplying X fragment j by
// the wave's 8 W fragments. The W fragments sit in registers for the block, the
// next block's are read into a second set while this one's MFMAs run (so blocks
// come in pairs: K a multiple of 256), and the X fragments stream three groups
// ahead of their MFMAs. Two barriers per block free the W and X halves of a stage
// for the copies of block j+2. On random operand codes the 16 x 16 x 128
// instruction reaches 0.88 of the nominal peak in a bare loop where the
// 32 x 32 x 64 one reaches 0.75 (the part is power-limited and the smaller
// instruction draws less per FLOP).
// LDS rows are 128 bytes; the 16-byte chunk c of row r sits at c ^ s(r) (see
// row_swizzle: conflict-free for the 16-row fragment reads).
//
// MFMA orientation: the instruction's A operand is the W tile (its rows are
// output channels n) and its B operand the X tile (columns are tokens m), so
// each lane's accumulators come in runs of 4 consecutive n of one m: the
// epilogue stores 8 bytes (4 bf16) per lane.
//
// Tile order: workgroup b runs on XCD b % 8; tiles are renumbered so each XCD
// walks a contiguous run of the tile space, grouped kGroupM (4) m-tiles at a time,
// which keeps the X and W slices its 32 CUs share resident in that XCD's L2.
//
// Every tile walks its K blocks in ascending order, so an output's bits do not depend on
// the tile it falls in. (Rotating the walk by one block in every second tile, or every second
// column of tiles, gave the same times: QKV 1.703 / 1.696 ms against 1.696 without, FFN-down
// 1.479 / 1.489 / 1.482, H3's shapes within 0.3%.)
//
// Shapes that would leave compute units idle go elsewhere, wholly or for their last round of
// tiles, as plan_gemm decides: to 224-row tiles of this kernel (XB = 7), to the smaller
// tiles of gemm_tile.hip -- which also take every K that is no multiple of 256 -- or, for
// rows of K >= 8192, to a split along K (units storing binary32 partial sums to a
// workspace, then k_gemm_splitk_reduce). A per-row gate and the residual apply in the fast
// epilogue's row layout (kEpiRowGate).
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "gemm_common.h"

namespace vdn {
namespace {

constexpr int BM = 256;        // tokens per tile
constexpr int BN = 256;        // output channels per tile
constexpr int kThreads = 256;  // 4 wavefronts, 2 (n) x 2 (m), 128 x 128 each
constexpr int kGroupM = 4;     // m-tiles per group of the tile order (GemmArgs::group_m)


// Internal epilogue (not an ABI value): VDN_FP8_EPI_GATE with a per-row gate index
// and/or a residual, on 16-byte rows -- the fast epilogue with the gate and the residual
// applied in the staging's row layout.
constexpr int kEpiRowGate = 4;


constexpr int64_t kUnitFloatsDev = 65536;   // floats of one split unit's partial sums (a 256 x 256 tile)

// Item v of a walk: whole tile v (v < t_main, all K blocks), or split unit v - t_main
// (blocks [kb0, kb0 + cnt) of its tile).
template <bool PARTIAL>
__device__ __forceinline__ void gemm_item(const GemmArgs& p, int nk, int v, int& tile, int& kb0, int& cnt, int& unit)
{
    if (!PARTIAL) {
        tile = v; kb0 = 0; cnt = nk; unit = -1;
    } else {
        // (integer division runs on the VALU: the results are made scalar again, as the
        // copies' inline assembly takes the block offset in an SGPR)
        unit = v - p.t_main;
        const int r = __builtin_amdgcn_readfirstlane(unit / p.splits);
        const int sl = unit - r * p.splits;
        tile = p.t_main + r;
        // (slice boundaries on even blocks: the K loop takes blocks two at a time)
        const int h = nk >> 1;
        kb0 = 2 * __builtin_amdgcn_readfirstlane(sl * h / p.splits);
        cnt = 2 * __builtin_amdgcn_readfirstlane((sl + 1) * h / p.splits) - kb0;
    }
}


// ---------------------------------------------------------------------------
// main kernel: K % 256 == 0, persistent
// ---------------------------------------------------------------------------

namespace mainloop {
constexpr int BK = 128;                     // K bytes per block (one LDS stage)
constexpr int kStage = (BM + BN) * BK;      // 64 KiB: X tile, then W tile
constexpr int kCopies = BN * BK / 1024 / 4; // 1 KiB copies of W per wave per block (8)
constexpr int kScal = 2 * kStage;           // per-tile vectors, two buffers of 4 x 1 KiB
constexpr int kStgRow = 144;                // epilogue staging row: 128 bytes + 16 of padding
constexpr int kStgWave = 32 * kStgRow;      // 32 rows per wave
constexpr int kStg = kScal + 8192;          // epilogue staging
constexpr int kLds = kStg + 4 * kStgWave;   // 154 KiB
constexpr int kStoreNT = 2;                 // cache policy of the output stores: non-temporal (the
                                            // output streams; keeps L2 for the operand panels)

__device__ __forceinline__ int lds_off(int row, int chunk) { return row * BK + ((chunk ^ row_swizzle(row)) << 4); }
}  // namespace mainloop


// Epilogue of the tile at (m0, n0) with its vectors in scalar buffer sb of smem
// acc[i][j][e] is n = wn*128 + 16 i + 4 (lane/16) + e, m = wm*128 + 16 j +
// lane%16 (tile-relative). Per 32-row band u and per 64-column half th the wave
// finishes its 32 x 64 slab (accumulators i = 4 th .. 4 th + 3, j = 2 u, 2 u + 1)
// in that layout (4 consecutive n per lane),
// writes it to its staging (32 rows of 128 bytes, padded to 144), reads it
// back by rows and stores 16-byte pieces of whole 128-byte row segments: lane
// L covers row 8 i + L/8, channels 8 (L%8) .. +7. The gate and residual
// apply in that row layout.
// The epilogue's slabs in order, for a wave of U bands: sidx = U (1 - th) + U - 1 - u,
// (th, u) = (1, U - 1), (1, U - 2), .. (0, 0). A slab mask (bit sidx; -1: every slab) restricts an epilogue to some of them.
constexpr bool slab_in(int mask, int s) { return mask < 0 || ((mask >> s) & 1); }
constexpr int slab_first(int mask) { return mask < 0 ? 0 : __builtin_ctz((unsigned)mask); }
constexpr int slab_last(int mask, int slabs) { return mask < 0 ? slabs - 1 : 31 - __builtin_clz((unsigned)mask); }

// scal: the tile's vectors (4 KiB: w_scale, x_scale, bias, gate index or gate row, 1 KiB
// each); stg: this wave's staging rows. Shared by the main kernel and the split-K reduction
// (four waves on a quadrant, each its 32 rows: MASK >= 0 restricts the epilogue to those
// slabs, bit sidx). XB: the wave's rows in sixteens.
template <int EPI, bool FAST, int MASK = -1, int XB = 8>
__device__ __forceinline__ void tile_epilogue(const GemmArgs& p, const uint8_t* scal, uint8_t* stg,
                                              f32x4_t (&acc)[8][XB], int64_t m0, int64_t n0, int wave)
{
    using namespace mainloop;
    static_assert(XB == 8 || MASK < 0, "slab masks are of the 256-row tile");
    constexpr int TM = 32 * XB, WM = 16 * XB;   // the tile's rows and the wave's
    constexpr int U = (XB + 1) / 2;             // 32-row bands of the wave (the last one 16 rows when XB is odd)
    const int wn = wave & 1, wm = wave >> 1;
    if constexpr (EPI == VDN_FP8_EPI_F32) {
        // binary32 (or binary16) rows, stored from the accumulators: 4 consecutive n of one m
        // per accumulator and lane; N % 4 == 0 keeps n .. n + 3 inside a row whenever n is
        uint32_t zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        const int el = (int)(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) + zero);
        const int fr = el & 15, fg = el >> 4;
        const float* s_sw = reinterpret_cast<const float*>(scal);
        const float* s_sx = reinterpret_cast<const float*>(scal + 1024);
        const bool half = p.out_type == VDN_FP8_DTYPE_F16, has_bias = p.bias != nullptr;
        float* out = reinterpret_cast<float*>(p.out);
#pragma unroll
        for (int j = 0; j < XB; ++j) {
            const int ml = wm * WM + 16 * j + fr;
            const int64_t m = m0 + ml;
            const float sxm = s_sx[ml];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (!slab_in(MASK, 4 * (1 - (i >> 2)) + 3 - (j >> 1))) continue;
                const int nl = wn * 128 + 16 * i + 4 * fg;
                const int64_t n = n0 + nl;
                const float4 sw = *reinterpret_cast<const float4*>(s_sw + nl);
                const float v[4] = {acc[i][j][0] * (sxm * sw.x), acc[i][j][1] * (sxm * sw.y),
                                    acc[i][j][2] * (sxm * sw.z), acc[i][j][3] * (sxm * sw.w)};
                if (m < p.M && n < p.N) {
                    if (half)
                        *reinterpret_cast<uint2*>(p.out + m * p.ldo + n) =
                            finish_f16x4(v, reinterpret_cast<const uint16_t*>(scal + 2048) + nl, has_bias);
                    else
                        *reinterpret_cast<float4*>(out + m * p.ldo + n) =
                            finish_f32x4(v, reinterpret_cast<const float*>(scal + 2048) + nl, has_bias);
                }
                acc[i][j] = f32x4_t{};   // the next tile starts from zero
            }
        }
        (void)stg;
        return;
    }
    const bool gate16 = ((p.ldgate & 7) == 0) && (((uintptr_t)p.gate & 15) == 0);
    const bool res16 = ((p.ldres & 7) == 0) && (((uintptr_t)p.residual & 15) == 0);
    // Every lane-dependent value here derives from an opaque zero, so the
    // compiler recomputes it per tile instead of holding it in registers
    // across the K loop.
    uint32_t zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
    const int el = (int)(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) + zero);
    const int fr = el & 15, fg = el >> 4, cc = el & 7, rl = el >> 3;
    const float* s_sw = reinterpret_cast<const float*>(scal);
    const float* s_sx = reinterpret_cast<const float*>(scal + 1024);
    const uint16_t* s_bias = reinterpret_cast<const uint16_t*>(scal + 2048);
    const int32_t* s_gi = reinterpret_cast<const int32_t*>(scal + 3072);
    const uint16_t* s_gate = reinterpret_cast<const uint16_t*>(scal + 3072);
    const __amdgpu_buffer_rsrc_t orr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.out + m0 * p.ldo), 0, (int)min(min(p.M - m0, (int64_t)TM) * p.ldo * 2, (int64_t)0x7fffffff), kRsrcWord3);
    const uint32_t ldo2 = (uint32_t)p.ldo * 2;
    // Slabs in order (th, u) = (1, 3), (1, 2), .. (0, 0). A column half's per-column
    // vectors (w_scale, bias and a broadcast gate row, unpacked to binary32) are read
    // from LDS once and held in registers across its four slabs -- the K loop's
    // fragment registers are free here. On the fast path the stores trail by one
    // slab: the previous slab's rows are read back from the staging before this
    // slab's values overwrite it (a wave's LDS operations run in order), so its
    // computation hides that read's latency.
    const bool has_bias = p.bias != nullptr;
    float hsw[4][4], hb[4][4], hg[4][4];
    auto hoist = [&](int th) {
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) {
            const int nl = wn * 128 + 64 * th + 16 * ii + 4 * fg;
            const float4 sw = *reinterpret_cast<const float4*>(s_sw + nl);
            hsw[ii][0] = sw.x; hsw[ii][1] = sw.y; hsw[ii][2] = sw.z; hsw[ii][3] = sw.w;
            if (has_bias) {
                const uint2 b = *reinterpret_cast<const uint2*>(s_bias + nl);
                hb[ii][0] = bf16_lo(b.x); hb[ii][1] = bf16_hi(b.x);
                hb[ii][2] = bf16_lo(b.y); hb[ii][3] = bf16_hi(b.y);
            }
            if (EPI == VDN_FP8_EPI_GATE && FAST) {
                const uint2 gv = *reinterpret_cast<const uint2*>(s_gate + nl);
                hg[ii][0] = bf16_lo(gv.x); hg[ii][1] = bf16_hi(gv.x);
                hg[ii][2] = bf16_lo(gv.y); hg[ii][3] = bf16_hi(gv.y);
            }
        }
    };
    // bf16 GEMM output, then the bf16 bias add: each rounding done two values per
    // conversion, the second one's pairs being the stored words (opaque, so the
    // compiler keeps the pairs); one uniform branch per slab
    auto compute = [&](int th, int u, auto with_bias) {
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            if (2 * u + jj >= XB) continue;
            const float sxm = s_sx[wm * WM + 32 * u + 16 * jj + fr];
#pragma unroll
            for (int ii = 0; ii < 4; ++ii) {
                const float* sw = hsw[ii];
                // A rounding to bf16 that the bias add or GELU reads is one conversion per
                // value (round_bf16_hi: no unpacking); the last one converts the stored
                // pairs. The gate kernels keep the packed pairs and unpack them (one value
                // per conversion there made the compiler spill).
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = acc[4 * th + ii][2 * u + jj][e] * (sxm * sw[e]);
                uint32_t r01, r23;
                if (EPI != VDN_FP8_EPI_GATE) {
                    if (decltype(with_bias)::value) {
                        const float* bb = hb[ii];
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = round_bf16_hi(v[e]) + bb[e];
                    }
                    if (EPI == VDN_FP8_EPI_GELU_TANH) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = gelu_tanh(round_bf16_hi(v[e]));   // of the bf16 output
                    }
                    r01 = pack_bf16x2(v[0], v[1]);
                    r23 = pack_bf16x2(v[2], v[3]);
                    asm volatile("" : "+v"(r01), "+v"(r23));
                } else {
                    r01 = pack_bf16x2(v[0], v[1]);
                    r23 = pack_bf16x2(v[2], v[3]);
                    asm volatile("" : "+v"(r01), "+v"(r23));
                    if (decltype(with_bias)::value) {
                        const float* bb = hb[ii];
                        r01 = pack_bf16x2(bf16_lo(r01) + bb[0], bf16_hi(r01) + bb[1]);
                        r23 = pack_bf16x2(bf16_lo(r23) + bb[2], bf16_hi(r23) + bb[3]);
                        asm volatile("" : "+v"(r01), "+v"(r23));
                    }
                    if (FAST) {   // broadcast gate row, no residual
                        const float* gg = hg[ii];
                        r01 = pack_bf16x2(bf16_lo(r01) * gg[0], bf16_hi(r01) * gg[1]);
                        r23 = pack_bf16x2(bf16_lo(r23) * gg[2], bf16_hi(r23) * gg[3]);
                    }
                }
                *reinterpret_cast<uint2*>(stg + (16 * jj + fr) * kStgRow + 32 * ii + 8 * fg) = make_uint2(r01, r23);
            }
        }
        // these accumulators start the next tile from zero
#pragma unroll
        for (int ii = 0; ii < 4; ++ii) {
            acc[4 * th + ii][2 * u] = f32x4_t{};
            if (2 * u + 1 < XB) acc[4 * th + ii][2 * u + 1] = f32x4_t{};
        }
    };
    // fast path: the slab's rows 8 i + L/8 from the staging, then their stores (byte
    // offset of the row, or out of range past N)
    uint4 pv[4];
    auto read_slab = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) pv[i] = *reinterpret_cast<const uint4*>(stg + (8 * i + rl) * kStgRow + (cc << 4));
    };
    // (the four offsets first, then the four stores back to back and their wait states)
    // Row gate: the gate table row gate_index[m] and the residual for the slab's rows
    // 8 i + L/8, columns 8 (L % 8) .. + 7 of the column half, by 16-byte buffer loads
    // issued two slabs ahead of their use into one of two register sets (rows past M and
    // columns past N read outside the descriptors: zeros), then, in the stores' row
    // layout, out = bf16(residual + gate * v) -- the gated residual kernel's arithmetic.
    constexpr bool kRowGate = EPI == kEpiRowGate;
    const bool has_res = p.residual != nullptr;
    const int64_t rows_here = min(p.M - m0, (int64_t)TM);
    const __amdgpu_buffer_rsrc_t rsr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(kRowGate && has_res ? p.residual + m0 * p.ldres : nullptr), 0,
        kRowGate && has_res ? (int)(((rows_here - 1) * p.ldres + p.N) * 2) : 0, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t gsr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(kRowGate ? p.gate : nullptr), 0, kRowGate ? (int)(((p.gate_rows - 1) * p.ldgate + p.N) * 2) : 0,
        kRsrcWord3);
    uint4 rres[2][4], rgat[2][4];
    auto load_rows = [&](int th, int u, int set) {
        const int64_t n = n0 + wn * 128 + 64 * th + 8 * cc;
        const bool nin = n < p.N;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (32 * u + 8 * i >= WM) continue;
            const int ml = wm * WM + 32 * u + 8 * i + rl;
            const int64_t gi = min(max((int64_t)s_gi[ml], (int64_t)0), p.gate_rows - 1);
            const uint32_t ro = nin ? (uint32_t)(((int64_t)ml * p.ldres + n) * 2) : 0x80000000u;
            const uint32_t go = nin ? (uint32_t)((gi * p.ldgate + n) * 2) : 0x80000000u;
            rres[set][i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsr, ro, 0, kBufferLoadOnce));
            rgat[set][i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(gsr, go, 0, 0));
        }
    };
    auto apply_rows = [&](int u, int set) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (32 * u + 8 * i >= WM) continue;
            const uint32_t vw[4] = {pv[i].x, pv[i].y, pv[i].z, pv[i].w};
            const uint32_t gw[4] = {rgat[set][i].x, rgat[set][i].y, rgat[set][i].z, rgat[set][i].w};
            const uint32_t rw[4] = {rres[set][i].x, rres[set][i].y, rres[set][i].z, rres[set][i].w};
            uint32_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // without a residual the product is stored as it is (no + 0: -0 stays -0)
                float lo = bf16_lo(gw[e]) * bf16_lo(vw[e]);
                float hi = bf16_hi(gw[e]) * bf16_hi(vw[e]);
                if (has_res) { lo = bf16_lo(rw[e]) + lo; hi = bf16_hi(rw[e]) + hi; }
                o[e] = pack_bf16x2(lo, hi);
            }
            pv[i] = make_uint4(o[0], o[1], o[2], o[3]);
        }
    };
    auto store_slab = [&](int th, int u, int set) {
        if constexpr (kRowGate) apply_rows(u, set);
        const int64_t n = n0 + wn * 128 + 64 * th + 8 * cc;
        const uint32_t off0 = (uint32_t)(wm * WM + 32 * u + rl) * ldo2 + (uint32_t)(n * 2);
        uint32_t off[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) off[i] = n < p.N ? off0 + (uint32_t)(8 * i) * ldo2 : 0x80000000u;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (32 * u + 8 * i < WM)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4_t, pv[i]), orr, off[i], 0, kStoreNT);
        settle_stores();
    };
    // (MASK >= 0: two slabs, kFirst and kLast)
    static_assert(MASK < 0 || __builtin_popcount((unsigned)MASK) == 2, "a slab mask holds two slabs");
    constexpr int kFirst = slab_first(MASK), kLast = slab_last(MASK, 2 * U);
    constexpr int kStep = MASK < 0 ? 1 : kLast - kFirst;
    // (the register set of slab sidx: the parity of its place in the order)
    auto set_of = [](int sidx) { return ((sidx - kFirst) / kStep) & 1; };
    if constexpr (kRowGate) load_rows(1 - kFirst / U, U - 1 - kFirst % U, 0);
#pragma unroll
    for (int sidx = 0; sidx < 2 * U; ++sidx) {
        const int th = 1 - sidx / U, u = U - 1 - sidx % U;
        if (MASK >= 0 && !((MASK >> sidx) & 1)) continue;
        if (MASK >= 0 || sidx % U == 0) hoist(th);
        if (FAST && sidx > kFirst) read_slab();   // the previous slab, before this one overwrites it
        if (has_bias) compute(th, u, std::true_type{});
        else compute(th, u, std::false_type{});
        if (FAST) {
            if (sidx > kFirst) store_slab(1 - (sidx - kStep) / U, U - 1 - (sidx - kStep) % U, set_of(sidx - kStep));
            if constexpr (kRowGate) {
                if (sidx < kLast) load_rows(1 - (sidx + kStep) / U, U - 1 - (sidx + kStep) % U, set_of(sidx + kStep));
            }
        } else {
            const int64_t n = n0 + wn * 128 + 64 * th + 8 * cc;
            const bool full = n + 8 <= p.N;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 8 * i + rl;
                if (32 * u + 8 * i >= WM) continue;
                uint4 v = *reinterpret_cast<const uint4*>(stg + r * kStgRow + (cc << 4));
                const int ml = wm * WM + 32 * u + r;
                const int64_t m = m0 + ml;
                if (m >= p.M || n >= p.N) continue;
                if (EPI == VDN_FP8_EPI_GATE) {
                    const int64_t gi = p.gate_index ? min(max((int64_t)s_gi[ml], (int64_t)0), p.gate_rows - 1) : 0;
                    const uint16_t* gp = p.gate + gi * p.ldgate + n;
                    uint4 g;
                    if (gate16 && full) g = *reinterpret_cast<const uint4*>(gp);
                    else {
                        const uint2 g0 = *reinterpret_cast<const uint2*>(gp);
                        const uint2 g1 = full ? *reinterpret_cast<const uint2*>(gp + 4) : make_uint2(0u, 0u);
                        g = make_uint4(g0.x, g0.y, g1.x, g1.y);
                    }
                    uint4 rv = make_uint4(0u, 0u, 0u, 0u);
                    if (p.residual) {
                        const uint16_t* rp = p.residual + m * p.ldres + n;
                        if (res16 && full) rv = *reinterpret_cast<const uint4*>(rp);
                        else {
                            const uint2 r0 = *reinterpret_cast<const uint2*>(rp);
                            const uint2 r1 = full ? *reinterpret_cast<const uint2*>(rp + 4) : make_uint2(0u, 0u);
                            rv = make_uint4(r0.x, r0.y, r1.x, r1.y);
                        }
                    }
                    const uint32_t vw[4] = {v.x, v.y, v.z, v.w}, gw[4] = {g.x, g.y, g.z, g.w},
                                   rw[4] = {rv.x, rv.y, rv.z, rv.w};
                    uint32_t o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float lo = bf16_lo(vw[e]) * bf16_lo(gw[e]), hi = bf16_hi(vw[e]) * bf16_hi(gw[e]);
                        if (p.residual) { lo += bf16_lo(rw[e]); hi += bf16_hi(rw[e]); }
                        o[e] = pack_bf16x2(lo, hi);
                    }
                    v = make_uint4(o[0], o[1], o[2], o[3]);
                }
                uint16_t* dst = p.out + m * p.ldo + n;
                *reinterpret_cast<uint2*>(dst) = make_uint2(v.x, v.y);
                if (full) *reinterpret_cast<uint2*>(dst + 4) = make_uint2(v.z, v.w);
            }
        }
        // one slab at a time: unbounded interleaving of slabs runs out of VGPRs
        __builtin_amdgcn_sched_barrier(0);
    }
    if (FAST) {   // the last slab
        read_slab();
        store_slab(1 - kLast / U, U - 1 - kLast % U, set_of(kLast));
    }
}

// One workgroup per CU walks tiles blockIdx.x, + gridDim.x, ... The copies form
// one stream of 128-byte K blocks across those tiles, so the next tile's first
// two blocks are in flight while this tile's epilogue runs. The block schedule
// (8 groups of 8 MFMAs, two barriers) is described at the K loop below.
// A tile's vectors (w_scale, x_scale, bias, gate rows) are copied into one of
// two scalar buffers at the start of the tile before, one copy per wave. The
// epilogue stages through LDS of its own.
//
// FAST (16-byte aligned output rows; a broadcast gate row travels with the tile's
// vectors, a per-row gate and the residual -- kEpiRowGate -- are loaded by the
// epilogue two slabs ahead of their use): the epilogue issues exactly 4 XB
// buffer stores per wave, columns past N sent out of range (dropped), and every
// load it issues has landed when it ends, so the waits that follow count the
// stores (conservatively, the counter retiring in issue order) and the stores
// drain while the next tile runs. Otherwise the waits also cover the epilogue's
// memory operations.
// PARTIAL: the split units instead of the whole tiles (one per workgroup, its K slice,
// the partial sums stored raw; a launch of its own, so that the whole-tile kernel keeps
// one straight-line epilogue; EPI and FAST do not matter to it: one instance serves).
template <int EPI, bool FAST, bool PARTIAL, int XB = 8>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
void k_gemm_fp8(GemmArgs p)
{
    using namespace mainloop;
    static_assert(XB == 8 || (XB == 7 && !PARTIAL), "256-row tiles, or whole 224-row ones");
    constexpr int TM = 32 * XB;                  // tokens per tile
    constexpr int kXCopies = XB, kWCopies = kCopies, kBlockCopies = kXCopies + kWCopies;   // per wave per block
    constexpr int kE = FAST ? 4 * XB : 0;        // 16-byte stores per wave per tile (fast epilogue)
    constexpr int XR = XB % 2 ? XB : 4;          // X fragments in rotation: two blocks are a whole number of turns
    __shared__ __attribute__((aligned(1024))) uint8_t smem[kLds];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave & 1, wm = wave >> 1;
    const int nk = (int)(p.K / BK);
    const int stride = gridDim.x;
    const int v_begin = PARTIAL ? p.t_main : 0;
    const int n_items = PARTIAL ? p.t_main + p.units : p.t_main;

    // Copies: this wave fills rows 64 wave .. 64 wave + 63 of each tile, 8 rows
    // (1 KiB) per copy. Lane L lands at row +L/8, physical chunk L%8, so it
    // fetches logical chunk (L%8) ^ row_swizzle(row), row = 64 wave + 8 i + L/8.
    // (recomputed per tile from an opaque lane index, with every other lane-dependent
    // value of the K loop, so that none is held in registers across the epilogue)
    uint32_t xoff[kXCopies], woff[kWCopies];
    auto opaque_lane = [&]() -> int {
        uint32_t zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        return (int)(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) + zero);
    };
    auto copy_offsets = [&](int l) {
#pragma unroll
        for (int i = 0; i < kWCopies; ++i) {
            const int r = 64 * wave + 8 * i + (l >> 3);
            const int c = (l & 7) ^ row_swizzle(r);
            woff[i] = (uint32_t)(r * p.ldw) + c * 16;
        }
#pragma unroll
        for (int i = 0; i < kXCopies; ++i) {
            const int r = 8 * XB * wave + 8 * i + (l >> 3);
            const int c = (l & 7) ^ row_swizzle(r);
            xoff[i] = (uint32_t)(r * p.ldx) + c * 16;
        }
    };
    copy_offsets(lane);
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void_t*)smem;

    // Producer: the next block to copy is block pj of item pv (pnk blocks; pkb its
    // first K byte). Blocks of items past the end still issue their copies, through
    // empty descriptors (zeros, no memory read), so the vmcnt bookkeeping stays fixed.
    int pv = v_begin + blockIdx.x, pj = 0, pkb = 0, pnk = nk;
    i32x4_t xr, wr;
    auto producer_tile = [&]() {
        int64_t xb = 0, wb = 0;
        const uint8_t* xa = p.xq;
        const uint8_t* wa = p.wq;
        pkb = 0;
        pnk = nk;
        if (pv < n_items) {
            int tile, kb0, unit, tm, tn;
            gemm_item<PARTIAL>(p, nk, pv, tile, kb0, pnk, unit);
            tile_coords(tile, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
            if (PARTIAL) pkb = kb0 * BK;
            const int64_t m0 = (int64_t)tm * TM, n0 = (int64_t)tn * BN;
            xa += m0 * p.ldx;
            wa += n0 * p.ldw;
            xb = min(p.M - m0, (int64_t)TM) * p.ldx;
            wb = min(p.N - n0, (int64_t)BN) * p.ldw;
        }
        xr = rsrc_words(xa, xb);
        wr = rsrc_words(wa, wb);
        asm volatile("s_nop 4");   // SGPR write by VALU -> use as a buffer descriptor
    };
    // Copy c of the producer's block into stage st: c < kWCopies is W rows 64 wave + 8 c ..,
    // else X rows.
    auto copy = [&](int st, int c) {
        const uint32_t dst = lds_base + (uint32_t)st * kStage;
        const uint32_t kb = (uint32_t)pkb;
        if (c < kWCopies) copy16_to_lds(wr, dst + BM * BK + (64 * wave + 8 * c) * BK, woff[c], kb);
        else copy16_to_lds(xr, dst + (8 * XB * wave + 8 * (c - kWCopies)) * BK, xoff[c - kWCopies], kb);
    };
    auto advance = [&]() {
        if (++pj == pnk) {
            pj = 0;
            pv += stride;
            producer_tile();
        } else {
            pkb += BK;
        }
    };
    // The vectors of the k-th tile of this workgroup go to scalar buffer k % 2:
    // wave 0 w_scale[n0 ..+255], wave 1 x_scale[m0 ..+255], wave 2 bias[n0 ..+511]
    // (256 used), wave 3 gate_index[m0 ..+255] -- or, for a broadcast gate on the
    // fast path, the gate row gate[0][n0 ..+511]. Missing ones read as zeros.
    auto scal_copy = [&](int t, int buf) {
        const void* base = p.sx;
        int64_t bytes = 0;
        if (t < p.t_main) {   // whole tiles only (split units store raw partial sums)
            int tm, tn;
            tile_coords(t, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
            const int64_t m0 = (int64_t)tm * TM, n0 = (int64_t)tn * BN;
            if (wave == 0) { base = p.sw + n0; bytes = min(p.N - n0, (int64_t)256) * 4; }
            else if (wave == 1) { base = p.sx + m0; bytes = min(p.M - m0, (int64_t)256) * 4; }
            else if (wave == 2) {
                const int64_t e = EPI == VDN_FP8_EPI_F32 && p.out_type == VDN_FP8_DTYPE_F32 ? 4 : 2;
                if (p.bias) { base = reinterpret_cast<const uint8_t*>(p.bias) + n0 * e; bytes = min((p.N - n0) * e, (int64_t)1024); }
            }
            else if (EPI == VDN_FP8_EPI_GATE && FAST) { base = p.gate + n0; bytes = min(p.N - n0, (int64_t)512) * 2; }
            else if (p.gate_index) { base = p.gate_index + m0; bytes = min(p.M - m0, (int64_t)256) * 4; }
        }
        const i32x4_t r = rsrc_words(base, bytes);
        asm volatile("s_nop 4");
        // the lane index recomputed here rather than kept live across the K loop
        uint32_t zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        const uint32_t l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) + zero;
        copy16_to_lds(r, lds_base + kScal + buf * 4096 + wave * 1024, l * 16, 0);
    };

    // acc[i][j] += W fragment i x X fragment j: 16 (n) x 16 (m) outputs over the whole block
    f32x4_t acc[8][XB];
    auto fence = [&]() { __builtin_amdgcn_sched_barrier(0); };

    auto epilogue = [&](int64_t m0, int64_t n0, int sb) {
        tile_epilogue<EPI, FAST, -1, XB>(p, smem + kScal + sb * 4096, smem + kStg + wave * kStgWave, acc, m0, n0, wave);
    };

    // Prologue: the first tile's vectors, then blocks 0 and 1 of the stream.
    producer_tile();
    scal_copy(v_begin + blockIdx.x, 0);
#pragma unroll
    for (int c = 0; c < kBlockCopies; ++c) copy(0, c);
    advance();
#pragma unroll
    for (int c = 0; c < kBlockCopies; ++c) copy(1, c);
    advance();

#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < XB; ++j) acc[i][j] = f32x4_t{};   // the epilogue re-zeroes them per tile
    int g = 0;    // stream index of the block being computed
    int k = 0;    // tiles done by this workgroup

    for (int v = v_begin + blockIdx.x; v < n_items; v += stride, ++k) {
        int tile, kb0, cnt, unit, tm, tn;
        gemm_item<PARTIAL>(p, nk, v, tile, kb0, cnt, unit);
        // (opaque: conditions on it are then evaluated per block, not hoisted out of
        // the tile loop into registers held across the epilogue)
        asm volatile("" : "+s"(cnt));
        tile_coords(tile, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
        const int64_t m0 = (int64_t)tm * TM, n0 = (int64_t)tn * BN;
        // Block g has landed once only block g+1's copies -- and, after the first
        // tile, the previous epilogue's stores -- may be pending.
        if (k == 0) wave_sync<kBlockCopies>();
        else wave_sync<kBlockCopies + kE>();
        scal_copy(v + stride, (k + 1) & 1);   // every wave is past the epilogue that used that buffer
        const int el = opaque_lane();
        copy_offsets(el);
        // Fragments of the block in stage st: 16 rows x 128 K bytes; lane L reads row
        // (base + L % 16), k bytes 32 (L / 16) .. +31, as two 16-byte chunks. W fragment
        // i is W rows wn*128 + 16 i .., X fragment j is X rows wm*128 + 16 j ..
        const int fr = el & 15, fg = el >> 4;
        auto read_frag = [&](const uint8_t* s, int row) -> i32x8_t {
            const uint4 lo = *reinterpret_cast<const uint4*>(s + lds_off(row, 2 * fg));
            const uint4 hi = *reinterpret_cast<const uint4*>(s + lds_off(row, 2 * fg + 1));
            return i32x8_t{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
        };
        auto read_w = [&](int st, int i) { return read_frag(smem + st * kStage + BM * BK, wn * 128 + 16 * i + fr); };
        auto read_x = [&](int st, int j) { return read_frag(smem + st * kStage, wm * 16 * XB + 16 * j + fr); };
        // W fragments of the block being computed and of the next one (read into the
        // other set while this block's MFMAs run); X fragments four at a time, in rotation.
        // (Declared per tile: nothing of them lives across the epilogue.)
        i32x8_t wa[8], wb[8], xf[XR];
        // Block g (j-th of the tile's cnt blocks, stage st = g % 2): 8 groups of 8 MFMAs,
        // group jx multiplying X fragment jx by the 8 W fragments.
        //   start (P0): W copies of block g+1 have landed in every wave, and every wave
        //     is done reading block g's W fragments (read during block g-1, or at the
        //     tile's start); group 1 then issues the W copies of block g+2 into stage st.
        //   group jx reads X fragment jx+3 (groups 5-7: block g+1's X fragments 0-2), three
        //     groups ahead of its MFMAs (one group ahead left them waiting on the read), and
        //     W fragment jx of block g+1.
        //   group 5 (P5): X copies of block g+1 have landed, every wave is done with block
        //     g's X fragments (the last read in group 4); groups 5 and 6 issue the X copies
        //     of block g+2 into stage st.
        // Copies newer than the awaited ones at P0 and P5: 8, plus in a tile's first block
        // the previous epilogue's stores and the vector copy. The tile's last block reads
        // the next one's fragments too (those of the next tile's first block, which the
        // next tile reads again): one code path, so the compiler's LDS waits count only
        // what each MFMA needs.
        // odd: which W set is current (wa in even blocks).
        auto kblock = [&](auto odd, int j) {
            i32x8_t (&wc)[8] = decltype(odd)::value ? wb : wa;
            i32x8_t (&wx)[8] = decltype(odd)::value ? wa : wb;
            const int st = g & 1;
            constexpr int xo = decltype(odd)::value ? XB % XR : 0;   // where this block's X fragments start
            // (newer copies at P0: the X copies of block g+1; at P5: the W copies of block g+2)
            auto sync = [&](auto newer) {
                constexpr int n = decltype(newer)::value;
                if (j > 0) wave_sync<n>();
                else if (k > 0) wave_sync<n + 1 + kE>();
                else wave_sync<n + 1>();
            };
            sync(std::integral_constant<int, kXCopies>{});
    #pragma unroll
            for (int jx = 0; jx < XB; ++jx) {
                if (jx == XB - 3) sync(std::integral_constant<int, kWCopies>{});
    #pragma unroll
                for (int i = 0; i < 8; ++i) {
                    acc[i][jx] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wc[i], xf[(jx + xo) % XR], acc[i][jx],
                                                                                   0, 0, 0, 0, 0, 0);
                    fence();
                    if (i == 0) xf[(jx + 3 + xo) % XR] = jx + 3 < XB ? read_x(st, jx + 3) : read_x(st ^ 1, jx + 3 - XB);
                    if (i == 4) {
                        wx[jx] = read_w(st ^ 1, jx);
                        if (XB == 7 && jx == 6) wx[7] = read_w(st ^ 1, 7);
                    }
                    // W copies of block g+2: two per group in groups 1 to 4 (224-row tiles, whose
                    // second barrier comes a group earlier: four in groups 1 and 2)
                    if (XB == 8) {
                        if (jx >= 1 && jx <= 4 && (i == 2 || i == 6)) copy(st, 2 * (jx - 1) + (i == 6));
                    } else {
                        if ((jx == 1 || jx == 2) && (i & 1)) copy(st, 4 * (jx - 1) + (i >> 1));
                    }
                    // X copies of block g+2
                    if ((jx == XB - 3 || jx == XB - 2) && (i & 1) && 4 * (jx - XB + 3) + (i >> 1) < kXCopies)
                        copy(st, kWCopies + 4 * (jx - XB + 3) + (i >> 1));
                    if (jx == XB - 2 && i == 7) advance();
                    fence();
                }
            }
            ++g;
        };

#pragma unroll
        for (int i = 0; i < 8; ++i) wa[i] = read_w(g & 1, i);
        xf[0] = read_x(g & 1, 0);
        xf[1] = read_x(g & 1, 1);
        xf[2] = read_x(g & 1, 2);
        // blocks 0, 1, .. cnt-1 (cnt even) alternate W sets (even: wa current)
        for (int j = 0; j < cnt; j += 2) {
            kblock(std::false_type{}, j);
            kblock(std::true_type{}, j + 1);
        }
        if constexpr (!PARTIAL) {
            epilogue(m0, n0, k & 1);
        } else {
            // (the launch has one workgroup per unit, so this is the workgroup's only item and
            // the accumulators are not re-zeroed)
            // A split unit stores its partial sums in accumulator layout: accumulator (i, j) of
            // lane L at (wave * 64 + 8 i + j) * 256 + 4 L of the unit's 65536 floats, one whole
            // KiB per wave store (a buffer descriptor over the wave's 64 KiB, four stores at a
            // time: the 256 accumulators are not all moved to VGPRs at once).
            const __amdgpu_buffer_rsrc_t wsr = __builtin_amdgcn_make_buffer_rsrc(
                (void*)(p.ws + ((int64_t)unit * 4 + wave) * 16384), 0, 65536, kRsrcWord3);
            uint32_t zero;
            asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
            const uint32_t l16 = (__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)) + zero) * 16;
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int j4 = 0; j4 < 2; ++j4) {
#pragma unroll
                    for (int jj = 0; jj < 4; ++jj) {
                        const int j = 4 * j4 + jj;
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4_t, acc[i][j]), wsr, l16,
                                                               (8 * i + j) * 1024, 0);
                    }
                    settle_stores();
                }
        }
    }
    // No copy may still be writing LDS when the workgroup ends.
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));
}

// The tile's vectors at (m0, n0) staged in LDS as the main kernel's copies lay them out
// (w_scale, x_scale, bias, then the broadcast gate row or gate_index), by one wave:
// branch-free buffer loads, all in flight at once; entries past N or M read as zeros.
template <int EPI, bool FAST>
__device__ __forceinline__ void stage_tile_vectors(const GemmArgs& p, uint8_t* scal, int64_t m0, int64_t n0, int lane)
{
    const int64_t nn = min(p.N - n0, (int64_t)256), mm = min(p.M - m0, (int64_t)256);
    const __amdgpu_buffer_rsrc_t swr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.sw + n0), 0, (int)(nn * 4), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t sxr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.sx + m0), 0, (int)(mm * 4), kRsrcWord3);
    const bool b32 = EPI == VDN_FP8_EPI_F32 && p.out_type == VDN_FP8_DTYPE_F32;   // a binary32 bias: 16 bytes per lane
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.bias ? p.bias + n0 * (b32 ? 2 : 1) : nullptr), 0, p.bias ? (int)(nn * (b32 ? 4 : 2)) : 0, kRsrcWord3);
    const bool grow = EPI == VDN_FP8_EPI_GATE && FAST;
    const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc(
        grow ? (void*)(p.gate + n0) : (void*)(p.gate_index ? p.gate_index + m0 : nullptr), 0,
        grow ? (int)(nn * 2) : (p.gate_index ? (int)(mm * 4) : 0), kRsrcWord3);
    const uint32_t l16 = (uint32_t)lane * 16, l8 = (uint32_t)lane * 8;
    const i32x4_t vsw = __builtin_amdgcn_raw_buffer_load_b128(swr, l16, 0, 0);
    const i32x4_t vsx = __builtin_amdgcn_raw_buffer_load_b128(sxr, l16, 0, 0);
    const i32x4_t vb4 = b32 ? __builtin_amdgcn_raw_buffer_load_b128(br, l16, 0, 0) : i32x4_t{};
    const i32x2_t vb = b32 ? i32x2_t{} : __builtin_amdgcn_raw_buffer_load_b64(br, l8, 0, 0);
    const i32x4_t vg4 = grow ? i32x4_t{} : __builtin_amdgcn_raw_buffer_load_b128(gr, l16, 0, 0);
    const i32x2_t vg2 = grow ? __builtin_amdgcn_raw_buffer_load_b64(gr, l8, 0, 0) : i32x2_t{};
    *reinterpret_cast<i32x4_t*>(scal + l16) = vsw;
    *reinterpret_cast<i32x4_t*>(scal + 1024 + l16) = vsx;
    if (b32) *reinterpret_cast<i32x4_t*>(scal + 2048 + l16) = vb4;
    else *reinterpret_cast<i32x2_t*>(scal + 2048 + l8) = vb;
    if (grow) *reinterpret_cast<i32x2_t*>(scal + 3072 + l8) = vg2;
    else *reinterpret_cast<i32x4_t*>(scal + 3072 + l16) = vg4;
}

// Split-K reduction: one workgroup of four waves per quadrant of a split tile (four per
// tile). Wave w sums accumulators 16 w .. 16 w + 15 of the quadrant (per lane) over the
// tile's units in slice order (slice 0 + slice 1 + ..., binary32: the order depends only
// on K and the split), two slices' loads in flight at once beside the sums, into LDS; wave
// 3 stages the tile's vectors as the main kernel's copies lay them out; then each wave
// runs the same epilogue for the quadrant's rows 32 w .. 32 w + 31 (its two slabs). Against
// one wave per quadrant holding all 64 accumulators: [3328, 5120, 8192] 0.124 -> 0.113 ms,
// [1000, 1000, 16384] 0.059 -> 0.042 ms, bitwise equal.
template <int EPI, bool FAST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void k_gemm_splitk_reduce(GemmArgs p)
{
    using namespace mainloop;
    __shared__ __attribute__((aligned(1024))) uint8_t scal[4096];
    __shared__ __attribute__((aligned(16))) uint8_t stg[4 * kStgWave];
    __shared__ f32x4_t sums[64 * 64];   // [accumulator][lane]
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int quad = blockIdx.x & 3, r = blockIdx.x >> 2;
    int tm, tn;
    tile_coords(p.t_main + r, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    if (w == 3) stage_tile_vectors<EPI, FAST>(p, scal, m0, n0, lane);
    const __amdgpu_buffer_rsrc_t wsr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(p.ws + (int64_t)r * p.splits * kUnitFloatsDev + (int64_t)quad * 16384), 0,
        (int)min((int64_t)p.splits * kUnitFloatsDev * 4, (int64_t)0x7fffffff), kRsrcWord3);
    const uint32_t l16 = (uint32_t)lane * 16;
    const int i0 = 16 * w;   // this wave's accumulators i0 .. i0 + 15
    f32x4_t a[16];
#pragma unroll
    for (int q = 0; q < 16; ++q)
        a[q] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(wsr, l16, (i0 + q) * 1024, 0));
    for (int sl = 1; sl < p.splits; sl += 2) {
        const bool two = sl + 1 < p.splits;
        // (a missing second slice is read past the descriptor's range: zeros, no traffic)
        const int so = sl * (int)kUnitFloatsDev * 4, so2 = so + (int)kUnitFloatsDev * 4;
        f32x4_t b[16], c[16];
#pragma unroll
        for (int q = 0; q < 16; ++q)
            b[q] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(wsr, l16, so + (i0 + q) * 1024, 0));
#pragma unroll
        for (int q = 0; q < 16; ++q)
            c[q] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(wsr, l16, so2 + (i0 + q) * 1024, 0));
#pragma unroll
        for (int q = 0; q < 16; ++q) a[q] += b[q];
        if (two) {
#pragma unroll
            for (int q = 0; q < 16; ++q) a[q] += c[q];
        }
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) sums[(i0 + q) * 64 + lane] = a[q];
    __syncthreads();
    // wave w: the epilogue's slabs of rows 32 w .. 32 w + 31 (accumulators [.][2 w], [.][2 w + 1])
    f32x4_t acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = sums[(8 * i + j) * 64 + lane];
    uint8_t* const ws = stg + w * kStgWave;
    switch (w) {
        case 0: tile_epilogue<EPI, FAST, 0x88>(p, scal, ws, acc, m0, n0, quad); break;
        case 1: tile_epilogue<EPI, FAST, 0x44>(p, scal, ws, acc, m0, n0, quad); break;
        case 2: tile_epilogue<EPI, FAST, 0x22>(p, scal, ws, acc, m0, n0, quad); break;
        default: tile_epilogue<EPI, FAST, 0x11>(p, scal, ws, acc, m0, n0, quad); break;
    }
}

// ---------------------------------------------------------------------------
// which kernels run a shape
// ---------------------------------------------------------------------------
// Split of the last partial round along K: for rows of at least 8192 bytes (K), when
// the tiles leave a last round of R <= grid / 2 tiles, each of those R tiles can run as S =
// min(grid / R, nk / 8) K slices on otherwise idle workgroups (at least 8 blocks each),
// then the reduction kernel sums the slices. The H3 FF down projection [13107, 5376,
// 14336]: 1092 tiles = 4 rounds + 68 on 256 CUs, the 68 as 3 slices of 37-38 blocks.
// Projections with shorter rows (the QKV and FF projections) never split: their outputs
// have the same bits whatever tiles they fall in, so a fused weight's outputs are those of
// its separate projections.
constexpr int64_t kSplitMinK = 8192;
constexpr int kSplitMinBlocks = 8;
constexpr int64_t kUnitFloats = 65536;   // one 256 x 256 tile of binary32 partial sums

// main: tiles 0 .. t_main - 1 (of 32 xb x 256) on the persistent kernel and, from t_main on,
// either `units` split units (with the reduction) or parts of (a, b) on the tile kernel;
// otherwise the tile kernel's (a, b) over the whole output.
struct GemmPlan {
    bool main;
    int xb, t_main, splits, units, a, b;
};

// The plan of a shape, by the estimated time of each way to run it, from rates measured on one
// MI355X, in us. Per 128-byte K block:
//   persistent kernel: a round of 256-row tiles 1.0 on a few compute units, 1.43 on all of
//     them (the part's power), of 224-row tiles 0.98 to 1.33;
//   tile kernel: kTiles' `alone`, or what the copies of all its tiles take at 16 TB/s out of
//     the L2s if that is longer; `busy` for a whole round of many; the weight's bytes at
//     4.9 TB/s bound the shortest calls;
//   a split: its slices' blocks at 1.2, and 14 us + 0.07 per slice for the partial sums and
//     their reduction.
// And per round the epilogue with its stores, which at a K of a few blocks is most of the time:
// 5.8 to 7.9 for 256-row tiles, 0.155 to 0.26 per 32 x 32 outputs of a tile of the tile kernel.
// Without that term shapes of K <= 1024 went to the tile kernel where the persistent one is
// faster: [2074, 10400, 256] 26.3 against 19.5 us, [1304, 2272, 1024] 12.1 against 9.9.
// Over 2143 drawn shapes (M 1 .. 16384, N 64 .. 30000, K 128 .. 16384, every epilogue, each way
// timed) the choice costs 1.5% on average against the best way, 9% at the 95th percentile;
// half of the estimates are within 9% of the time, nine tenths between 0.75 and 1.24 of it.
// [821, 5376, 5120], 84 tiles of 256 x 256 on 256 CUs: 47 us there, 27.3 us as 196 tiles of
// 192 channels x 128 tokens; [300, 5376, 5120] 31 -> 17.6 us; [1299, 28672, 5376] 180 -> 172 us
// with 224-row tiles (the same 672 tiles, an eighth less of each); [4680, 13824, 5120] 260 -> 246.
GemmPlan plan_gemm(int64_t M, int64_t N, int64_t K, int cus, bool split_ok, bool rows224_ok, double* est = nullptr)
{
    const double nk = (double)((K + mainloop::BK - 1) / mainloop::BK);
    int count = 0;
    const GemmTile* tiles = gemm_tiles(&count);
    const double floor_us = (double)N * (double)K / 4.9e6 + 3.0;
    auto part_us = [&](const GemmTile& t, double units) {   // at most one round of them
        const double copies = units * (t.a + t.b) * 4096e-6 / 16.0;
        const double epilogue = (0.155 + 0.05 * std::min(1.0, units / cus)) * t.a * t.b;
        return std::max(nk * std::max(t.alone, copies) + 3.2 + epilogue, floor_us);
    };
    auto tile_of = [&](int a, int b) {
        int i = 0;
        while (tiles[i].a != a || tiles[i].b != b) ++i;
        return tiles[i];
    };
    GemmPlan best{};
    double best_us = 1e30;
    auto take = [&](double us, const GemmPlan& p) {
        if (us < best_us) { best_us = us; best = p; }
    };
    if (K % (2 * mainloop::BK) == 0) {
        const int64_t tn = (N + BN - 1) / BN;
        for (int xb = 8; xb >= (rows224_ok ? 7 : 8); --xb) {
            const int64_t T = ((M + 32 * xb - 1) / (32 * xb)) * tn, full = T / cus, R = T % cus;
            auto round_us = [&](double load) {
                return nk * (xb == 8 ? 1.0 + 0.43 * load : 0.98 + 0.35 * load) + (xb == 8 ? 5.8 + 2.1 * load : 4.8 + 1.7 * load);
            };
            const double base = (double)full * round_us(1.0) + (full ? 5.0 : 0.0);
            const GemmPlan whole{true, xb, (int)T, 0, 0, 0, 0};
            if (R == 0) { take(base, whole); continue; }
            if (xb == 8) {
                const int64_t S = 2 * R <= cus ? std::min<int64_t>(cus / R, (int64_t)nk / kSplitMinBlocks) : 0;
                if (split_ok && K >= kSplitMinK && S >= 2) {
                    const double split_us = base + nk / (double)S * 1.2 + 14.0 + 0.07 * (double)(R * S);
                    const GemmPlan split{true, 8, (int)(T - R), (int)S, (int)(R * S), 0, 0};
                    // At most 16 tiles always split, so that the size query's answer for such an output
                    // stays what it has been. On one MI355X, split against whole chains of small
                    // tiles (what a call without a workspace runs): [256, 4096, 28672] 52 / 101 us,
                    // [1024, 1024, 32768] 48 / 62, [300, 512, 14336] 30 / 32, [1024, 1024, 14336] 36 / 33, but
                    // [1000, 1024, 8192] 31 / 19 and [300, 512, 8192] 25 / 19.
                    if (T <= 16) {
                        if (est) *est = split_us;
                        return split;
                    }
                    take(split_us, split);
                }
                if (2 * R <= cus) take(base + part_us(tile_of(8, 4), 2.0 * (double)R) + 0.4, {true, 8, (int)(T - R), 0, 0, 8, 4});
                if (4 * R <= cus) take(base + part_us(tile_of(4, 4), 4.0 * (double)R) + 0.4, {true, 8, (int)(T - R), 0, 0, 4, 4});
                // (a last round of so few tiles is bound by one part's chain of K blocks, and this part's
                // block is the shortest: [4680, 13824, 5120], two tiles left of 1026, 244.6 us as
                // quarters, 238.8 as eighths. Longer rows split along K.)
                if (8 * R <= cus && K < kSplitMinK)
                    take(base + part_us(tile_of(4, 2), 8.0 * (double)R) + 0.4, {true, 8, (int)(T - R), 0, 0, 4, 2});
            }
            take(base + round_us((double)R / cus) + (full ? 0.0 : 5.0), whole);
        }
    }
    for (int i = 0; i < count; ++i) {
        const GemmTile& t = tiles[i];
        const int64_t units = ((M + 32 * t.b - 1) / (32 * t.b)) * ((N + 32 * t.a - 1) / (32 * t.a));
        double us = (double)(units / cus) * (nk * t.busy + 0.26 * t.a * t.b);
        us += units % cus ? part_us(t, (double)(units % cus)) : 5.0;
        take(K >= kSplitMinK ? 1.1 * us : us, {false, 0, 0, 0, 0, t.a, t.b});
    }
    if (est) *est = best_us;
    return best;
}

// The plan of a call. The workspace's size is asked for by M, N and K alone, as for 16-byte rows, so
// other rows split only where that answer holds the partial sums: a workspace of the answered
// size is never too small. ([2900, 28672, 8192]: 224-row tiles and no workspace for 16-byte rows,
// where other rows alone would be estimated fastest as 256 slices, 64 MiB.)
GemmPlan plan_call(int64_t M, int64_t N, int64_t K, int cus, bool workspace, bool rows16, double* est = nullptr)
{
    const bool split_ok = workspace && K >= kSplitMinK && (rows16 || plan_gemm(M, N, K, cus, true, true).units);
    return plan_gemm(M, N, K, cus, split_ok, rows16, est);
}

}  // namespace

int launch_gated_residual(const uint16_t* residual, int64_t ldr, const uint16_t* gate, int64_t ldgate,
                          const int32_t* gate_index, int64_t gate_rows, const uint16_t* branch, int64_t ldb,
                          uint16_t* out, int64_t ldo, int64_t M, int64_t N, hipStream_t stream);

// Bytes of split-K workspace a [M, N, K] GEMM takes on the current device (0: no split).
int gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t* bytes)
{
    *bytes = 0;
    if (M <= 0 || N <= 0 || K <= 0) return VDN_FP8_OK;
    const int cus = device_cus();
    if (cus <= 0) return set_error(VDN_FP8_ELAUNCH, "gemm: cannot query the device's compute units");
    const int64_t T = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
    if (T > (int64_t)INT32_MAX / 16) return VDN_FP8_OK;
    *bytes = (int64_t)plan_call(M, N, K, cus, true, true).units * kUnitFloats * (int64_t)sizeof(float);
    return VDN_FP8_OK;
}

// The GEMM with an optional split-K workspace (ws NULL: no split). out_type: VDN_FP8_DTYPE_F16
// or _F32 with VDN_FP8_EPI_F32 (bias of that type); -1: what the epilogue implies.
int gemm_launch(const void* xq, const float* x_scale, const void* wq, const float* w_scale, int64_t M, int64_t N,
                int64_t K, int64_t ldx, int64_t ldw, const void* bias, int epilogue, const void* gate,
                const int32_t* gate_index, int64_t gate_rows, int64_t ldgate, const void* residual, int64_t ldres,
                void* out, int64_t ldo, float* ws, int64_t ws_bytes, hipStream_t stream, int out_type)
{
    if (M < 0 || N < 0 || K < 0) return set_error(VDN_FP8_EINVAL, "gemm: negative shape");
    if (M == 0 || N == 0) return VDN_FP8_OK;
    if (K == 0 || K % 16) return set_error(VDN_FP8_EINVAL, "gemm: K must be a positive multiple of 16 (K=%lld)", (long long)K);
    if (N % 4) return set_error(VDN_FP8_EINVAL, "gemm: N must be a multiple of 4 (N=%lld)", (long long)N);
    if (!xq || !wq || !x_scale || !w_scale || !out) return set_error(VDN_FP8_EINVAL, "gemm: null pointer");
    if (ldx < K || ldw < K || ldo < N || ldx % 16 || ldw % 16 || ldo % 4)
        return set_error(VDN_FP8_EINVAL, "gemm: need ldx, ldw >= K and multiples of 16, ldo >= N and a multiple of 4");
    if (ldx * 256 > (int64_t)0x7fffffff || ldw * 256 > (int64_t)0x7fffffff)
        return set_error(VDN_FP8_EINVAL, "gemm: row stride too large (256 rows must span < 2 GiB)");
    if (!aligned(xq, 16) || !aligned(wq, 16) || !aligned(out, 8) || !aligned(w_scale, 16) || !aligned(x_scale, 16) ||
        (bias && !aligned(bias, 16)) || (gate_index && !aligned(gate_index, 16)))
        return set_error(VDN_FP8_EINVAL, "gemm: misaligned operand (xq, wq, x_scale, w_scale, bias, gate_index 16 B; out 8 B)");
    if (epilogue == VDN_FP8_EPI_GATE) {
        if (!gate || gate_rows < 1) return set_error(VDN_FP8_EINVAL, "gemm: the gate epilogue needs a gate table of >= 1 row");
        if (ldgate < N || ldgate % 4 || !aligned(gate, 8)) return set_error(VDN_FP8_EINVAL, "gemm: gate rows must be >= N and 8-byte aligned");
        if (residual && (ldres < N || ldres % 4 || !aligned(residual, 8)))
            return set_error(VDN_FP8_EINVAL, "gemm: residual rows must be >= N and 8-byte aligned");
    } else if (epilogue == VDN_FP8_EPI_F32) {
        if ((bias && out_type < 0) || gate || residual || gate_index)
            return set_error(VDN_FP8_EINVAL, "gemm: the binary32 output takes no bias, gate or residual");
        if (out_type != VDN_FP8_DTYPE_F16 && !aligned(out, 16)) return set_error(VDN_FP8_EINVAL, "gemm: the binary32 output must be 16-byte aligned");
    } else if (epilogue != VDN_FP8_EPI_NONE && epilogue != VDN_FP8_EPI_GELU_TANH) {
        return set_error(VDN_FP8_EINVAL, "gemm: unknown epilogue %d", epilogue);
    }
    if (ws_bytes < 0 || (ws && !aligned(ws, 16))) return set_error(VDN_FP8_EINVAL, "gemm: workspace must be 16-byte aligned");
    const int64_t tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN, T = tiles_m * tiles_n;
    if (T > (int64_t)INT32_MAX / 16) return set_error(VDN_FP8_EINVAL, "gemm: problem too large");
    const int cus = device_cus();
    if (cus <= 0) return set_error(VDN_FP8_ELAUNCH, "gemm: cannot query the device's compute units");
    // The fast epilogue: 16-byte output rows, row offsets within 31 bits; a gate table and
    // a residual on 16-byte rows too. A broadcast gate row is staged like the bias
    // (VDN_FP8_EPI_GATE); a per-row gate or a residual applies in the epilogue's row layout
    // (kEpiRowGate: bf16(residual + gate[i] * v), the gated residual kernel's arithmetic; H3 FF
    // down [13107, 5376, 14336] with a gate table and the residual: 0.750 -> 0.691 ms against
    // the GEMM writing v and that kernel reading it back; bitwise equal).
    const int64_t kMax = 0x7fffffff;
    const bool gated = epilogue == VDN_FP8_EPI_GATE;
    const bool out16 = N % 8 == 0 && ldo % 8 == 0 && aligned(out, 16) && (int64_t)BM * ldo * 2 <= kMax;
    const bool gate_broadcast = gated && !residual && (gate_rows == 1 || !gate_index) && aligned(gate, 16);
    const bool rows16 = gated && out16 && aligned(gate, 16) && ldgate % 8 == 0 &&
                        (!residual || (aligned(residual, 16) && ldres % 8 == 0));
    const bool rows31 = rows16 && (!residual || (int64_t)BM * ldres * 2 <= kMax) && gate_rows * ldgate * 2 <= kMax;
    const bool fast = out16 && epilogue != VDN_FP8_EPI_F32 && (!gated || gate_broadcast || rows31);
    const GemmPlan plan = plan_call(M, N, K, cus, ws != nullptr, fast);
    GemmArgs p{(const uint8_t*)xq, x_scale, (const uint8_t*)wq, w_scale, M, N, K, ldx, ldw,
               (const uint16_t*)bias, (const uint16_t*)gate, gate_index, gate_rows, ldgate,
               (const uint16_t*)residual, ldres, (uint16_t*)out, ldo,
               epilogue == VDN_FP8_EPI_F32 && out_type < 0 ? VDN_FP8_DTYPE_F32 : std::max(out_type, 0), (int)tiles_m, (int)tiles_n,
               kGroupM, plan.t_main, plan.splits, plan.units, ws};
    const bool tile_fast = out16 && (!gated || rows31);
    const int64_t part_m = plan.main ? 1 : (M + 32 * plan.b - 1) / (32 * plan.b), part_n = plan.main ? 1 : (N + 32 * plan.a - 1) / (32 * plan.a);
    if (part_m * part_n >= 1 << 24) {
        // A launch of 2^24 workgroups passes 2^32 work-items, of which HIP starts only the remainder:
        // two halves, each planned by itself. (Here rather than by a second grid dimension, whose
        // index cost the tile kernel 0.5 us of [821, 5376, 5120]'s 27.)
        const int64_t hm = part_m >= part_n ? (M / 2 + 255) / 256 * 256 : 0, hn = hm ? 0 : (N / 2 + 255) / 256 * 256;
        const int64_t be = p.out_type == VDN_FP8_DTYPE_F32 ? 4 : 2;   // bytes of a bias value and of an output
        for (int h = 0; h < 2; ++h) {
            const int64_t m0 = h ? hm : 0, n0 = h ? hn : 0;
            auto at = [](const void* t, int64_t off) { return t ? (const void*)((const uint8_t*)t + off) : nullptr; };
            const int st = gemm_launch(p.xq + m0 * ldx, x_scale + m0, p.wq + n0 * ldw, w_scale + n0,
                                       hm ? (h ? M - hm : hm) : M, hn ? (h ? N - hn : hn) : N, K, ldx, ldw, at(bias, n0 * be), epilogue,
                                       at(gate, n0 * 2), (const int32_t*)at(gate_index, m0 * 4), gate_rows, ldgate,
                                       at(residual, (m0 * ldres + n0) * 2), ldres, (uint8_t*)out + (m0 * ldo + n0) * be, ldo, nullptr, 0,
                                       stream, out_type);
            if (st != VDN_FP8_OK) return st;
        }
        return VDN_FP8_OK;
    }
    if (!plan.main) return launch_gemm_tile(p, plan.a, plan.b, 0, epilogue, tile_fast, stream);
    const int64_t need = (int64_t)plan.units * kUnitFloats * (int64_t)sizeof(float);
    if (ws_bytes < need)
        return set_error(VDN_FP8_EINVAL, "gemm: workspace of %lld bytes, this shape needs %lld", (long long)ws_bytes,
                         (long long)need);
    p.tiles_m = (int)((M + 32 * plan.xb - 1) / (32 * plan.xb));
    const int rest = plan.a ? (int)(T - plan.t_main) : 0;   // 256 x 256 tiles for the tile kernel
    const dim3 grid((unsigned)std::min(plan.t_main, cus)), block(kThreads);
    const dim3 ugrid((unsigned)plan.units), rgrid((unsigned)(plan.units ? 4 * (plan.units / plan.splits) : 0));
#define VDN_MAIN(E, F)                                                                                    \
    do {                                                                                                  \
        if (p.t_main) hipLaunchKernelGGL((k_gemm_fp8<E, F, false>), grid, block, 0, stream, p);           \
        if (p.units) {                                                                                    \
            hipLaunchKernelGGL((k_gemm_fp8<VDN_FP8_EPI_NONE, true, true>), ugrid, block, 0, stream, p);   \
            hipLaunchKernelGGL((k_gemm_splitk_reduce<E, F>), rgrid, dim3(256), 0, stream, p);             \
        }                                                                                                 \
        if (rest) {                                                                                       \
            const int st = launch_gemm_tile(p, plan.a, plan.b, rest, epilogue, tile_fast, stream);        \
            if (st != VDN_FP8_OK) return st;                                                              \
        }                                                                                                 \
    } while (0)
#define VDN_MAIN_FAST(E)                                                                                  \
    do {                                                                                                  \
        if (plan.xb == 7) hipLaunchKernelGGL((k_gemm_fp8<E, true, false, 7>), grid, block, 0, stream, p); \
        else VDN_MAIN(E, true);                                                                           \
    } while (0)
    if (rows16 && !rows31 && !gate_broadcast) {
        // rows whose offsets pass 31 bits: the GEMM writing v, then the gated residual kernel
        const int st = gemm_launch(xq, x_scale, wq, w_scale, M, N, K, ldx, ldw, bias, VDN_FP8_EPI_NONE, nullptr, nullptr,
                                   0, 0, nullptr, 0, out, ldo, ws, ws_bytes, stream, -1);
        if (st != VDN_FP8_OK) return st;
        return launch_gated_residual((const uint16_t*)residual, ldres, (const uint16_t*)gate, ldgate, gate_index,
                                     gate_rows, (const uint16_t*)out, ldo, (uint16_t*)out, ldo, M, N, stream);
    }
    if (epilogue == VDN_FP8_EPI_F32) {
        VDN_MAIN(VDN_FP8_EPI_F32, false);   // (the general epilogue only: the fast one stages bf16 rows)
    } else if (gated && !gate_broadcast && fast) {
        VDN_MAIN_FAST(kEpiRowGate);
    } else if (gated) {
        if (fast) VDN_MAIN_FAST(VDN_FP8_EPI_GATE);
        else VDN_MAIN(VDN_FP8_EPI_GATE, false);
    } else if (epilogue == VDN_FP8_EPI_GELU_TANH) {
        if (fast) VDN_MAIN_FAST(VDN_FP8_EPI_GELU_TANH);
        else VDN_MAIN(VDN_FP8_EPI_GELU_TANH, false);
    } else {
        if (fast) VDN_MAIN_FAST(VDN_FP8_EPI_NONE);
        else VDN_MAIN(VDN_FP8_EPI_NONE, false);
    }
#undef VDN_MAIN_FAST
#undef VDN_MAIN
    return check_launch("gemm");
}
}  // namespace vdn

using namespace vdn;

extern "C" int vdn_fp8_gemm(const void* xq, const float* x_scale, const void* wq, const float* w_scale, int64_t M,
                            int64_t N, int64_t K, int64_t ldx, int64_t ldw, const void* bias, int epilogue,
                            const void* gate, const int32_t* gate_index, int64_t gate_rows, int64_t ldgate,
                            const void* residual, int64_t ldres, void* out, int64_t ldo, hipStream_t stream)
{
    return gemm_launch(xq, x_scale, wq, w_scale, M, N, K, ldx, ldw, bias, epilogue, gate, gate_index, gate_rows,
                       ldgate, residual, ldres, out, ldo, nullptr, 0, stream, -1);
}

extern "C" int vdn_fp8_gemm_workspace_size(int64_t M, int64_t N, int64_t K, int64_t* bytes)
{
    if (!bytes) return set_error(VDN_FP8_EINVAL, "gemm_workspace_size: null pointer");
    return gemm_workspace_bytes(M, N, K, bytes);
}

extern "C" int vdn_fp8_gemm_plan(int64_t M, int64_t N, int64_t K, int rows16, int workspace, int cus, int32_t* plan,
                                 double* us)
{
    if (!plan) return set_error(VDN_FP8_EINVAL, "gemm_plan: null pointer");
    if (M <= 0 || N <= 0 || K <= 0 || cus < 0) return set_error(VDN_FP8_EINVAL, "gemm_plan: sizes must be positive");
    if (((M + BM - 1) / BM) * ((N + BN - 1) / BN) > (int64_t)INT32_MAX / 16)
        return set_error(VDN_FP8_EINVAL, "gemm_plan: problem too large");
    if (cus == 0 && (cus = device_cus()) <= 0)
        return set_error(VDN_FP8_ELAUNCH, "gemm_plan: cannot query the device's compute units");
    const GemmPlan p = plan_call(M, N, K, cus, workspace != 0, rows16 != 0, us);
    const int32_t v[6] = {p.main ? 32 * p.xb : 0, p.main ? p.t_main : 0, p.units ? p.splits : 0, p.units, 32 * p.a, 32 * p.b};
    for (int i = 0; i < 6; ++i) plan[i] = v[i];
    return VDN_FP8_OK;
}

extern "C" int vdn_fp8_gemm_ws(const void* xq, const float* x_scale, const void* wq, const float* w_scale, int64_t M,
                               int64_t N, int64_t K, int64_t ldx, int64_t ldw, const void* bias, int epilogue,
                               const void* gate, const int32_t* gate_index, int64_t gate_rows, int64_t ldgate,
                               const void* residual, int64_t ldres, void* out, int64_t ldo, void* workspace,
                               int64_t workspace_bytes, hipStream_t stream)
{
    return gemm_launch(xq, x_scale, wq, w_scale, M, N, K, ldx, ldw, bias, epilogue, gate, gate_index, gate_rows,
                       ldgate, residual, ldres, out, ldo, (float*)workspace, workspace_bytes, stream, -1);
}

extern "C" int vdn_fp8_gemm_typed(const void* xq, const float* x_scale, const void* wq, const float* w_scale, int64_t M,
                                  int64_t N, int64_t K, int64_t ldx, int64_t ldw, const void* bias, int dtype, void* out,
                                  int64_t ldo, void* workspace, int64_t workspace_bytes, hipStream_t stream)
{
    if (dtype != VDN_FP8_DTYPE_F16 && dtype != VDN_FP8_DTYPE_F32)
        return set_error(VDN_FP8_EINVAL, "gemm_typed: the output is binary16 or binary32 (dtype %d)", dtype);
    return gemm_launch(xq, x_scale, wq, w_scale, M, N, K, ldx, ldw, bias, VDN_FP8_EPI_F32, nullptr, nullptr, 0, 0, nullptr,
                       0, out, ldo, (float*)workspace, workspace_bytes, stream, dtype);
}

// ---------------------------------------------------------------------------
// The allocation-free GEMM: the split-K workspace in a static device array
// ---------------------------------------------------------------------------
// Largest split workspace on a 256-CU part: units <= compute units, 256 KiB each.
constexpr int64_t kScratchBytes = 64LL << 20;
static __device__ __align__(256) float scratch[kScratchBytes / sizeof(float)];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch[kMaxScratchDevices];   // this device's copy of `scratch`, or null before the first call

// The device address of `scratch` on the current device, looked up on the first call on
// each device (the host-side name is not a device address); null if the lookup fails.
float* scratch_ptr(int dev)
{
    if (dev < 0 || dev >= kMaxScratchDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
            (void)hipGetLastError();
            return nullptr;
        }
        g_scratch[dev] = static_cast<float*>(ptr);
    }
    return g_scratch[dev];
}
}  // namespace

extern "C" int vdn_fp8_gemm_noalloc(const void* xq, const float* x_scale, const void* wq, const float* w_scale,
                                    int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, const void* bias,
                                    int epilogue, const void* gate, const int32_t* gate_index, int64_t gate_rows,
                                    int64_t ldgate, const void* residual, int64_t ldres, void* out, int64_t ldo,
                                    hipStream_t stream)
{
    int64_t need = 0;
    const int st = gemm_workspace_bytes(M, N, K, &need);
    if (st != VDN_FP8_OK) return st;
    if (need > kScratchBytes)
        return set_error(VDN_FP8_EINVAL, "gemm_noalloc: this shape's split workspace (%lld bytes) exceeds the "
                                         "static scratch of %lld bytes", (long long)need, (long long)kScratchBytes);
    float* ws = nullptr;
    if (need > 0) {
        int dev = -1;
        if (hipGetDevice(&dev) != hipSuccess) return set_error(VDN_FP8_ELAUNCH, "gemm_noalloc: no current device");
        ws = scratch_ptr(dev);
        if (!ws) return set_error(VDN_FP8_ELAUNCH, "gemm_noalloc: cannot look up the scratch array on device %d", dev);
    }
    return gemm_launch(xq, x_scale, wq, w_scale, M, N, K, ldx, ldw, bias, epilogue, gate, gate_index, gate_rows,
                       ldgate, residual, ldres, out, ldo, ws, ws ? kScratchBytes : 0, stream, -1);
}
