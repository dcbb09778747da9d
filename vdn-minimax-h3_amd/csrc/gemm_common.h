// What the GEMM's kernels share: the problem's arguments, the tile order, global -> LDS
// copies with their waits, and the LDS row swizzle.
#pragma once

#include <stdint.h>

#include "vdn_common.h"

namespace vdn {

constexpr int kRsrcWord3 = 0x00020000;   // raw buffer, 32-bit data format (gfx9 family)

typedef int i32x2_t __attribute__((ext_vector_type(2)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void_t;

struct GemmArgs {
    const uint8_t* xq;
    const float* sx;
    const uint8_t* wq;
    const float* sw;
    int64_t M, N, K, ldx, ldw;
    const uint16_t* bias;   // of the output's type (out_type)
    const uint16_t* gate;
    const int32_t* gate_index;
    int64_t gate_rows, ldgate;
    const uint16_t* residual;
    int64_t ldres;
    uint16_t* out;
    int64_t ldo;
    int out_type;           // VDN_FP8_DTYPE_*: binary16 and binary32 with VDN_FP8_EPI_F32
    int tiles_m, tiles_n;
    int group_m;   // m-tiles per group of the tile order
    // Split of the last partial round along K (long rows only): the first t_main tiles
    // (in tile order) run whole; each of the others runs as `splits` K slices, unit u
    // being slice u % splits of tile t_main + u / splits, whose fp32 partial sums go to
    // ws (65536 floats per unit, accumulator layout) and are summed by the reduction
    // kernel, slice by slice, before the epilogue. units = 0: no split (t_main = T).
    int t_main, splits, units;
    float* ws;
};

// One tile shape of the tile kernel (gemm_tile.hip), 32 a channels x 32 b tokens, and its time
// in us per 128-byte K block, alone on the part and with every compute unit busy.
struct GemmTile {
    int a, b;
    double alone, busy;
};
const GemmTile* gemm_tiles(int* count);

// The tile kernel over the whole output (rest = 0), or over the last `rest` 256 x 256 tiles
// from p.t_main on (a and b 4 or 8). epilogue: the C ABI's; fast: 16-byte rows throughout.
int launch_gemm_tile(GemmArgs p, int a, int b, int rest, int epilogue, bool fast, hipStream_t stream);

// Four outputs of a binary16 or binary32 row (VDN_FP8_EPI_F32): the binary32 product in the
// output's type, then the bias of that type, rounded where the reference's cast and `out +
// bias` round. b: the four bias values in LDS.
__device__ __forceinline__ uint2 finish_f16x4(const float (&v)[4], const uint16_t* b, bool has_bias)
{
    _Float16 h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float t = v[e];
        asm volatile("" : "+v"(t));   // rounded to binary32 first (else one instruction multiplies and rounds to binary16)
        h[e] = (_Float16)t;
        if (has_bias) h[e] = (_Float16)((float)h[e] + (float)__builtin_bit_cast(_Float16, b[e]));
    }
    auto pair = [](_Float16 lo, _Float16 hi) {
        return (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
    };
    return make_uint2(pair(h[0], h[1]), pair(h[2], h[3]));
}

__device__ __forceinline__ float4 finish_f32x4(const float (&v)[4], const float* b, bool has_bias)
{
    if (!has_bias) return make_float4(v[0], v[1], v[2], v[3]);
    return make_float4(v[0] + b[0], v[1] + b[1], v[2] + b[2], v[3] + b[3]);
}

// Renumbers workgroup b so that XCD (b % 8) gets a contiguous run of tiles,
// then maps the run index to (tile_m, tile_n) in groups of gm m-tiles.
__device__ __forceinline__ void tile_coords(int b, int tiles_m, int tiles_n, int gm, int& tm, int& tn)
{
    const int T = tiles_m * tiles_n;
    const int q = T / 8, r = T % 8, xcd = b % 8, local = b / 8;
    const int t = (xcd < r) ? xcd * (q + 1) + local : r * (q + 1) + (xcd - r) * q + local;
    const int group = gm * tiles_n;
    const int first_m = (t / group) * gm;
    const int gsize = min(tiles_m - first_m, gm);
    tm = first_m + (t % group) % gsize;
    tn = (t % group) / gsize;
}

// One wave-wide 16-byte-per-lane copy global -> LDS: lane L's 16 bytes at
// buffer offset voff + soff land at LDS byte lds + 16 L. Written as inline
// assembly so that the compiler does not treat every later LDS read as
// dependent on it (it would wait for all such copies, serializing the
// pipeline); the kernel waits on vmcnt itself. M0 carries the LDS address and
// is restored afterwards; s_nop covers the M0-write -> LDS-DMA hazard.
__device__ __forceinline__ void copy16_to_lds(i32x4_t rsrc, uint32_t lds, uint32_t voff, uint32_t soff)
{
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %2, %3, %4 offen lds\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
        : "memory");
}

// s_waitcnt immediates (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] << 14)
constexpr int waitcnt_vm_lgkm0(int vm) { return (vm & 15) | (7 << 4) | (0 << 8) | ((vm >> 4) << 14); }

// This wave's copies, except the VM most recent, have landed and its LDS reads
// are done; then all waves meet. The scheduling barriers keep the compiler from
// moving instructions across (MFMAs touch no memory and would otherwise float).
template <int VM>
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(VM));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// Row r, 16-byte chunk c (0..7) of a 128-byte-row LDS tile sits at chunk c ^ s(r),
// s(r) = bits 1, 0, 2 of r. A 16 x 128-byte fragment read (lane L: row L % 16, chunk
// 2 (L / 16), then the next chunk) runs without bank conflicts under this swizzle --
// measured over every XOR swizzle of the row's low four bits: 1342 of the 4096 run at
// the full rate, the XOR with bits 1..3 of the row (conflict-free for the 32-row reads
// of the 32 x 32 x 64 instruction) at half of it.
__device__ __forceinline__ int row_swizzle(int row) { return ((row >> 1) & 1) | ((row & 1) << 1) | (row & 4); }

// Buffer descriptor (raw, 32-bit data format, gfx9 family) over `bytes` bytes from base: reads past
// them are zeros. Wave-uniform, in SGPRs.
__device__ __forceinline__ i32x4_t rsrc_words(const void* base, int64_t bytes)
{
    const uint64_t a = (uint64_t)base;
    bytes = max(min(bytes, (int64_t)0x7fffffff), (int64_t)0);
    return i32x4_t{__builtin_amdgcn_readfirstlane((int)(a & 0xffffffffu)),
                   __builtin_amdgcn_readfirstlane((int)((a >> 32) & 0xffffu)),
                   __builtin_amdgcn_readfirstlane((int)bytes), kRsrcWord3};
}

}  // namespace vdn
