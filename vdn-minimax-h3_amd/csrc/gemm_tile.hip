// The fp8 GEMM for shapes whose 256 x 256 tiles leave compute units idle, and for every K
// that the persistent kernel does not take (gemm.hip: K a multiple of 256): one output tile
// of 32 A channels x 32 B tokens per workgroup, A and B chosen so that the tiles fill the
// part. Same arithmetic as the persistent kernel -- one chain of
// v_mfma_f32_16x16x128_f8f6f4 per output over the 128-byte K blocks in ascending order, the
// same rounding points after it -- so an output has the same bits whatever tile it falls in.
//
// A workgroup of 4 waves, 2 (n) x 2 (m), 16 A x 16 B outputs each. K advances in 128-byte
// blocks through a ring of S LDS stages ((A + B) x 4 KiB each) filled by global -> LDS
// copies; both operands' fragments are double-buffered in registers: while block g's MFMAs
// run, block g + 1's fragments are read, so block g's stage is free at the block's start
// (one barrier) and takes the copies of block g + S at once. S - 1 blocks are in flight:
// with one or two tiles per compute unit nothing else hides the copies' latency, which at
// ~0.7 us is two to four blocks of these tiles.
// K % 128 != 0: in the last block the lanes whose 16 bytes lie past K copy from outside
// the descriptor (zeros).
#include "gemm_common.h"

namespace vdn {
namespace {

constexpr int kThreads = 256;
constexpr int BK = 128;

template <int A, int B, int S>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
void k_gemm_tile(GemmArgs p, int epi, int fast)
{
    constexpr int TN = 32 * A, TM = 32 * B;        // channels, tokens of the tile
    constexpr int kStage = (A + B) * 4096;         // TM X rows, then TN W rows, of 128 bytes
    constexpr int C = A + B;                       // 1 KiB copies per wave per block
    constexpr int RS = 32 * A + 16;                // epilogue staging row: the wave's 16 A channels, padded
    constexpr int kScal = S * kStage;              // w_scale, x_scale, bias, gate_index of the tile, 1 KiB each
    static_assert(4 * 16 * B * RS <= S * kStage, "the epilogue stages where the blocks were");
    static_assert(C * (S - 1) + 1 <= 63, "the wait counts fit the counter");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[kScal + 4096];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wn = wave & 1, wm = wave >> 1;
    const int nk = (int)((p.K + BK - 1) / BK);
    int tm, tn;
    int64_t m0, n0;
    if (p.t_main < 0) {
        tile_coords(blockIdx.x, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
        m0 = (int64_t)tm * TM;
        n0 = (int64_t)tn * TN;
    } else {
        // the 256 x 256 tiles from t_main on (the persistent kernel's order) in (8 / A) (8 / B) parts
        constexpr int PN = 8 / A, PM = 8 / B;
        const int part = blockIdx.x % (PN * PM);
        tile_coords(p.t_main + (int)(blockIdx.x / (PN * PM)), p.tiles_m, p.tiles_n, p.group_m, tm, tn);
        m0 = (int64_t)tm * 256 + (part / PN) * TM;
        n0 = (int64_t)tn * 256 + (part % PN) * TN;
        if (m0 >= p.M || n0 >= p.N) return;
    }
    const int64_t rows_here = min(p.M - m0, (int64_t)TM);

    // The tile's vectors, one copy per wave (entries past N or M, and missing vectors, zeros).
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_void_t*)smem;
    {
        const void* base = p.sx;
        int64_t bytes = 0;
        if (wave == 0) { base = p.sw + n0; bytes = min(p.N - n0, (int64_t)256) * 4; }
        else if (wave == 1) { base = p.sx + m0; bytes = min(p.M - m0, (int64_t)256) * 4; }
        else if (wave == 2) {
            const int64_t e = p.out_type == VDN_FP8_DTYPE_F32 ? 4 : 2;   // bytes of a bias value
            if (p.bias) { base = reinterpret_cast<const uint8_t*>(p.bias) + n0 * e; bytes = min((p.N - n0) * e, (int64_t)1024); }
        }
        else if (p.gate_index) { base = p.gate_index + m0; bytes = min(p.M - m0, (int64_t)256) * 4; }
        const i32x4_t r = rsrc_words(base, bytes);
        asm volatile("s_nop 4");   // SGPR write by VALU -> use as a buffer descriptor
        copy16_to_lds(r, lds_base + kScal + wave * 1024, (uint32_t)lane * 16, 0);
    }

    // Copies: this wave fills 8 B X rows and 8 A W rows of a stage, 8 rows (1 KiB) per copy;
    // lane L lands at row + L/8, physical chunk L%8, so it fetches logical chunk
    // (L%8) ^ row_swizzle(row) (the swizzle of a row is that of L/8: the rows before it
    // are multiples of 8).
    i32x4_t xr = rsrc_words(p.xq + m0 * p.ldx, rows_here * p.ldx);
    i32x4_t wr = rsrc_words(p.wq + n0 * p.ldw, min(p.N - n0, (int64_t)TN) * p.ldw);
    asm volatile("s_nop 4");
    const int xbytes = xr[2], wbytes = wr[2];
    const int chunk16 = ((lane & 7) ^ row_swizzle(lane >> 3)) << 4;
    uint32_t xoff[B], woff[A];
#pragma unroll
    for (int i = 0; i < B; ++i) xoff[i] = (uint32_t)((8 * B * wave + 8 * i + (lane >> 3)) * p.ldx) + chunk16;
#pragma unroll
    for (int i = 0; i < A; ++i) woff[i] = (uint32_t)((8 * A * wave + 8 * i + (lane >> 3)) * p.ldw) + chunk16;
    // Copy c of block kb into stage st; blocks past the last one still issue theirs, through
    // empty descriptors (zeros, no memory read), so that the counts the waits rely on hold. (The
    // part adds the scalar offset before it compares with the range, and does not wrap: copies
    // of a zero range at scalar offsets inside a buffer gave zeros.)
    auto copy = [&](uint32_t st, int kb, int c) {
        const bool out = kb * BK + chunk16 >= (int)p.K;   // this lane's 16 bytes lie past K
        const int live = kb < nk ? -1 : 0;
        if (c < B) {
            xr[2] = xbytes & live;
            copy16_to_lds(xr, st + (8 * B * wave + 8 * c) * BK, out ? 0x80000000u : xoff[c], (uint32_t)(kb * BK));
        } else {
            wr[2] = wbytes & live;
            copy16_to_lds(wr, st + TM * BK + (8 * A * wave + 8 * (c - B)) * BK, out ? 0x80000000u : woff[c - B],
                          (uint32_t)(kb * BK));
        }
    };
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int c = 0; c < C; ++c) copy(lds_base + s * kStage, s, c);

    // Fragments: 16 rows x 128 K bytes, lane L row L % 16, bytes 32 (L / 16) .. + 31 as two
    // 16-byte chunks.
    const int fr = lane & 15, fg = lane >> 4;
    const int lo = fr * BK + (((2 * fg) ^ row_swizzle(fr)) << 4), hi = fr * BK + (((2 * fg + 1) ^ row_swizzle(fr)) << 4);
    auto read_frag = [&](const uint8_t* s) -> i32x8_t {
        const uint4 a = *reinterpret_cast<const uint4*>(s + lo);
        const uint4 b = *reinterpret_cast<const uint4*>(s + hi);
        return i32x8_t{(int)a.x, (int)a.y, (int)a.z, (int)a.w, (int)b.x, (int)b.y, (int)b.z, (int)b.w};
    };
    i32x8_t wf[2][A], xf[2][B];
    auto read_one = [&](auto set, int st, int f) {   // fragment f of a stage: X fragments, then W fragments
        constexpr int s = decltype(set)::value;
        const uint8_t* base = smem + st * kStage;
        if (f < B) xf[s][f] = read_frag(base + (16 * B * wm + 16 * f) * BK);
        else wf[s][f - B] = read_frag(base + TM * BK + (16 * A * wn + 16 * (f - B)) * BK);
    };
    f32x4_t acc[A][B];
#pragma unroll
    for (int i = 0; i < A; ++i)
#pragma unroll
        for (int j = 0; j < B; ++j) acc[i][j] = f32x4_t{};

    wave_sync<(S - 1) * C>();   // block 0 (and the vectors) landed
#pragma unroll
    for (int f = 0; f < C; ++f) read_one(std::integral_constant<int, 0>{}, 0, f);
    int st = 0;                 // block g's stage
    // Block g: every wave has read block g's fragments (its stage is free) and block g + 1 has
    // landed; then its MFMAs, among them the reads of block g + 1's fragments and the
    // copies of block g + S.
    auto kblock = [&](auto set, int g) {
        constexpr int s = decltype(set)::value;
        wave_sync<(S - 2) * C>();
        const int nx = st + 1 == S ? 0 : st + 1;
        const uint32_t dst = lds_base + (uint32_t)st * kStage;
#pragma unroll
        for (int q = 0; q < A * B; ++q) {
            const int j = q / A, i = q % A;
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf[s][i], xf[s][j], acc[i][j], 0, 0, 0, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (q < C) read_one(std::integral_constant<int, 1 - s>{}, nx, q);
#pragma unroll
            for (int c = 0; c < C; ++c)
                if (c * A * B / C == q) copy(dst, g + S, c);
            __builtin_amdgcn_sched_barrier(0);
        }
        st = nx;
    };
    for (int g = 0; g < nk; g += 2) {
        kblock(std::integral_constant<int, 0>{}, g);
        if (g + 1 < nk) kblock(std::integral_constant<int, 1>{}, g + 1);
    }
    wave_sync<0>();   // no copy is in flight and no wave reads a stage: the staging may overlay them

    // Epilogue. acc[i][j][e] is channel 16 A wn + 16 i + 4 fg + e of token 16 B wm + 16 j + fr.
    const float* s_sw = reinterpret_cast<const float*>(smem + kScal);
    const float* s_sx = reinterpret_cast<const float*>(smem + kScal + 1024);
    const uint16_t* s_bias = reinterpret_cast<const uint16_t*>(smem + kScal + 2048);
    const int32_t* s_gi = reinterpret_cast<const int32_t*>(smem + kScal + 3072);
    const bool has_bias = p.bias != nullptr;
    if (epi == VDN_FP8_EPI_F32 && p.out_type == VDN_FP8_DTYPE_F32) {   // binary32 rows, from the accumulators
        float* out = reinterpret_cast<float*>(p.out);
        const float* s_bf = reinterpret_cast<const float*>(smem + kScal + 2048);
#pragma unroll
        for (int j = 0; j < B; ++j) {
            const int ml = 16 * (B * wm + j) + fr;
            const float sxm = s_sx[ml];
#pragma unroll
            for (int i = 0; i < A; ++i) {
                const int nl = 16 * (A * wn + i) + 4 * fg;
                const float4 sw = *reinterpret_cast<const float4*>(s_sw + nl);
                const float v[4] = {acc[i][j][0] * (sxm * sw.x), acc[i][j][1] * (sxm * sw.y),
                                    acc[i][j][2] * (sxm * sw.z), acc[i][j][3] * (sxm * sw.w)};
                if (m0 + ml < p.M && n0 + nl < p.N)
                    *reinterpret_cast<float4*>(out + (m0 + ml) * p.ldo + n0 + nl) = finish_f32x4(v, s_bf + nl, has_bias);
            }
        }
        return;
    }
    uint8_t* const stg = smem + wave * 16 * B * RS;
    // the wave's 16 B x 16 A outputs, rounded where the reference rounds (a missing bias adds
    // -0, which leaves every value as it is), into its own staging rows
    auto finish = [&](auto gelu, auto half) {
#pragma unroll
        for (int i = 0; i < A; ++i) {
            const int nl = 16 * (A * wn + i) + 4 * fg;
            const float4 sw = *reinterpret_cast<const float4*>(s_sw + nl);
            const uint2 b = *reinterpret_cast<const uint2*>(s_bias + nl);
            const float b0 = has_bias ? bf16_lo(b.x) : -0.0f, b1 = has_bias ? bf16_hi(b.x) : -0.0f;
            const float b2 = has_bias ? bf16_lo(b.y) : -0.0f, b3 = has_bias ? bf16_hi(b.y) : -0.0f;
#pragma unroll
            for (int j = 0; j < B; ++j) {
                const float sxm = s_sx[16 * (B * wm + j) + fr];
                if (decltype(half)::value) {
                    const float v[4] = {acc[i][j][0] * (sxm * sw.x), acc[i][j][1] * (sxm * sw.y),
                                        acc[i][j][2] * (sxm * sw.z), acc[i][j][3] * (sxm * sw.w)};
                    *reinterpret_cast<uint2*>(stg + (16 * j + fr) * RS + 32 * i + 8 * fg) = finish_f16x4(v, s_bias + nl, has_bias);
                    continue;
                }
                uint32_t r01 = pack_bf16x2(acc[i][j][0] * (sxm * sw.x), acc[i][j][1] * (sxm * sw.y));
                uint32_t r23 = pack_bf16x2(acc[i][j][2] * (sxm * sw.z), acc[i][j][3] * (sxm * sw.w));
                asm volatile("" : "+v"(r01), "+v"(r23));   // each pair in one conversion
                r01 = pack_bf16x2(bf16_lo(r01) + b0, bf16_hi(r01) + b1);
                r23 = pack_bf16x2(bf16_lo(r23) + b2, bf16_hi(r23) + b3);
                asm volatile("" : "+v"(r01), "+v"(r23));
                if (decltype(gelu)::value) {
                    r01 = pack_bf16x2(gelu_tanh(bf16_lo(r01)), gelu_tanh(bf16_hi(r01)));
                    r23 = pack_bf16x2(gelu_tanh(bf16_lo(r23)), gelu_tanh(bf16_hi(r23)));
                }
                *reinterpret_cast<uint2*>(stg + (16 * j + fr) * RS + 32 * i + 8 * fg) = make_uint2(r01, r23);
            }
        }
    };
    if (epi == VDN_FP8_EPI_GELU_TANH) finish(std::true_type{}, std::false_type{});
    else if (epi == VDN_FP8_EPI_F32) finish(std::false_type{}, std::true_type{});   // binary16 rows
    else finish(std::false_type{}, std::false_type{});
    // out = bf16(residual + gate[i] * v) on packed pairs, in the rows' layout
    const bool gated = epi == VDN_FP8_EPI_GATE, has_res = p.residual != nullptr;
    auto gate_pair = [&](uint32_t v, uint32_t g, uint32_t r) {
        float a = bf16_lo(g) * bf16_lo(v), b = bf16_hi(g) * bf16_hi(v);
        if (has_res) { a = bf16_lo(r) + a; b = bf16_hi(r) + b; }
        return pack_bf16x2(a, b);
    };
    if (fast) {
        // 16-byte pieces, 2 A of them per row: whole row segments per store, rows past M and
        // columns past N outside the descriptors (loads zero, stores dropped)
        constexpr int kPieces = A * B / 2;   // per lane
        const __amdgpu_buffer_rsrc_t orr = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(p.out + m0 * p.ldo), 0, (int)min(rows_here * p.ldo * 2, (int64_t)0x7fffffff), kRsrcWord3);
        const __amdgpu_buffer_rsrc_t rsr = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(has_res ? p.residual + m0 * p.ldres : nullptr), 0,
            has_res ? (int)(((rows_here - 1) * p.ldres + p.N) * 2) : 0, kRsrcWord3);
        const __amdgpu_buffer_rsrc_t gsr = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(gated ? p.gate : nullptr), 0, gated ? (int)(((p.gate_rows - 1) * p.ldgate + p.N) * 2) : 0, kRsrcWord3);
        auto pieces = [&](auto with_gate) {
            constexpr bool kGate = decltype(with_gate)::value;
#pragma unroll
            for (int it0 = 0; it0 < kPieces; it0 += 4) {
                uint4 v[4], g[4], r[4];
                uint32_t off[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (it0 + u >= kPieces) continue;
                    const int idx = (it0 + u) * 64 + lane, row = idx / (2 * A), pc = idx % (2 * A);
                    const int ml = 16 * B * wm + row;
                    const int64_t n = n0 + 16 * A * wn + 8 * pc;
                    v[u] = *reinterpret_cast<const uint4*>(stg + row * RS + pc * 16);
                    off[u] = n < p.N ? (uint32_t)ml * (uint32_t)(p.ldo * 2) + (uint32_t)(n * 2) : 0x80000000u;
                    if (kGate) {
                        const int64_t gi = min(max((int64_t)s_gi[ml], (int64_t)0), p.gate_rows - 1);
                        const uint32_t ro = n < p.N ? (uint32_t)(((int64_t)ml * p.ldres + n) * 2) : 0x80000000u;
                        const uint32_t go = n < p.N ? (uint32_t)((gi * p.ldgate + n) * 2) : 0x80000000u;
                        r[u] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rsr, ro, 0, kBufferLoadOnce));
                        g[u] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(gsr, go, 0, 0));
                    }
                }
                if (kGate) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (it0 + u >= kPieces) continue;
                        v[u] = make_uint4(gate_pair(v[u].x, g[u].x, r[u].x), gate_pair(v[u].y, g[u].y, r[u].y),
                                          gate_pair(v[u].z, g[u].z, r[u].z), gate_pair(v[u].w, g[u].w, r[u].w));
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (it0 + u < kPieces)
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4_t, v[u]), orr, off[u], 0, 0);
                settle_stores();
            }
        };
        if (gated) pieces(std::true_type{});
        else pieces(std::false_type{});
        return;
    }
    // other rows: 8-byte pieces, 4 A of them per row
    for (int idx = lane; idx < 16 * B * 4 * A; idx += 64) {
        const int row = idx / (4 * A), pc = idx % (4 * A);
        const int64_t m = m0 + 16 * B * wm + row, n = n0 + 16 * A * wn + 4 * pc;
        if (m >= p.M || n >= p.N) continue;
        uint2 v = *reinterpret_cast<const uint2*>(stg + row * RS + pc * 8);
        if (gated) {
            const int64_t gi = min(max((int64_t)s_gi[16 * B * wm + row], (int64_t)0), p.gate_rows - 1);
            const uint2 g = *reinterpret_cast<const uint2*>(p.gate + gi * p.ldgate + n);
            const uint2 r = has_res ? *reinterpret_cast<const uint2*>(p.residual + m * p.ldres + n) : make_uint2(0u, 0u);
            v = make_uint2(gate_pair(v.x, g.x, r.x), gate_pair(v.y, g.y, r.y));
        }
        *reinterpret_cast<uint2*>(p.out + m * p.ldo + n) = v;
    }
}

// Tile shapes, in 32-channel and 32-token units, with their stages: as many as the LDS holds
// (five and four where latency counts most), at most 512 registers' worth of accumulators and
// two sets of fragments (8 x 5 already moves fragments through AGPRs: 47 against 33 us for
// 8 x 4 on [821, 5376, 5120]).
#define VDN_TILES(X) X(4, 2, 5) X(4, 3, 5) X(4, 4, 4) X(4, 6, 3) X(6, 3, 4) X(6, 4, 3) X(8, 4, 3)

// Measured on one MI355X, in us per 128-byte K block. alone: a tile with most compute units
// idle (its copies and MFMAs); busy: 256 tiles round after round (their copies share the
// L2s and the part's power).
constexpr GemmTile kTiles[] = {{4, 2, 0.27, 0.42}, {4, 3, 0.305, 0.56}, {4, 4, 0.345, 0.62}, {4, 6, 0.47, 0.80},
                               {6, 3, 0.40, 0.75}, {6, 4, 0.48, 0.85}, {8, 4, 0.64, 1.0}};

}  // namespace

const GemmTile* gemm_tiles(int* count)
{
    *count = (int)(sizeof(kTiles) / sizeof(kTiles[0]));
    return kTiles;
}

int launch_gemm_tile(GemmArgs p, int a, int b, int rest, int epilogue, bool fast, hipStream_t stream)
{
    unsigned units;
    if (rest > 0) {
        units = (unsigned)(rest * (8 / a) * (8 / b));
    } else {
        p.t_main = -1;
        p.tiles_m = (int)((p.M + 32 * b - 1) / (32 * b));
        p.tiles_n = (int)((p.N + 32 * a - 1) / (32 * a));
        units = (unsigned)p.tiles_m * (unsigned)p.tiles_n;
    }
    const dim3 grid(units), block(kThreads);
#define VDN_TILE_LAUNCH(A, B, S)                                                                          \
    if (a == A && b == B) {                                                                               \
        hipLaunchKernelGGL((k_gemm_tile<A, B, S>), grid, block, 0, stream, p, epilogue, (int)fast);       \
        return check_launch("gemm");                                                                      \
    }
    VDN_TILES(VDN_TILE_LAUNCH)
#undef VDN_TILE_LAUNCH
    return set_error(VDN_FP8_ELAUNCH, "gemm: no kernel of %d x %d tiles", 32 * b, 32 * a);
}

}  // namespace vdn
