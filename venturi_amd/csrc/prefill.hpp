// Shared parts of the prefill GEMMs (more than 32 tokens): tile order and
// tiling choice on the host, LDS swizzle, register slots, lane offsets and the
// final sum over the waves that split K.
//
// Two kernel forms use them. The cooperative one stages a tile's operands in
// LDS for a whole workgroup, whose waves split the tile and the K range of a
// stage (one 32-column group per K wave); the split one gives every wave of a
// workgroup the same small tile and its own share of K with an LDS region of
// its own, so that its main loop has no barrier.
#pragma once

#include "common.hpp"

#include <type_traits>
#include <utility>

namespace vt {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));

// Tile order: workgroups are dealt to the 8 XCDs round robin, so XCD b % 8
// takes a contiguous run of tiles in which the token tiles of one weight tile
// follow each other: a weight tile is fetched into one XCD's L2 and shared
// there (W8A16, 512 tokens x 34816 rows, 64 x 64 tiles: 395 -> 336 us against
// token tiles in grid.y; 128 tokens: 121 -> 108).
struct TileOrder {
    int token_tiles, tiles, per_xcd;
};

inline TileOrder tile_order(int tokens, int tm, int n, int tn) {
    TileOrder o;
    o.token_tiles = (tokens + tm - 1) / tm;
    const std::int64_t tiles = static_cast<std::int64_t>(o.token_tiles) * ((n + tn - 1) / tn);
    require(tiles <= INT32_MAX - 8, "tiles exceed the launch grid");
    o.tiles = static_cast<int>(tiles);
    o.per_xcd = static_cast<int>((tiles + 7) / 8);
    return o;
}

// The workgroup's tile, or -1 past the last one.
__device__ __forceinline__ int tile_of(const TileOrder& o) {
    const int slot = static_cast<int>(blockIdx.x >> 3);
    const int tile = static_cast<int>(blockIdx.x & 7) * o.per_xcd + slot;
    return tile < o.tiles ? tile : -1;
}

// A tiling's measured time model, in microseconds: every round of workgroups
// costs `round` (prologue, sum over the K waves, output) plus, per 1024
// columns, `solo` when it leaves at most one workgroup on a CU, `full` when a
// CU holds `per_cu`, and in proportion between; `base` once.
struct PrefillTiling {
    int tm, tn, per_cu;
    double base, round, solo, full;
};

inline double tiling_time(const PrefillTiling& t, int tokens, int n, double k) {
    const std::int64_t tiles = static_cast<std::int64_t>((tokens + t.tm - 1) / t.tm) * ((n + t.tn - 1) / t.tn);
    const std::int64_t slots = static_cast<std::int64_t>(device_cus()) * t.per_cu;
    const std::int64_t whole = tiles / slots, rest = tiles % slots;
    const std::int64_t level = (rest + device_cus() - 1) / device_cus();  // workgroups on a CU in the last round
    const double last = level == 0 ? 0.0 : level == 1 ? t.solo : t.solo + (t.full - t.solo) * static_cast<double>(level - 1) / (t.per_cu - 1);
    return t.base + static_cast<double>(whole + (rest > 0)) * t.round + k / 1024.0 * (static_cast<double>(whole) * t.full + last);
}

template <int N>
inline int fastest_tiling(const PrefillTiling (&tilings)[N], int tokens, int n, double k) {
    int best = 0;
    for (int i = 1; i < N; ++i)
        if (tiling_time(tilings[i], tokens, n, k) < tiling_time(tilings[best], tokens, n, k)) best = i;
    return best;
}

// XOR swizzle of the 16-byte units of a staged row of U units, so that the
// same unit of 16 consecutive rows falls on 16 distinct 16-byte bank groups.
template <int U>
__device__ __forceinline__ int swizzle(int row) {
    if constexpr (U >= 16) return row & 15;
    else return (row / (16 / U)) & (U - 1);
}

// Compile-time register slots: every stage in flight keeps its own registers.
template <int P>
using Slot = std::integral_constant<int, P>;

template <class F, int... P>
__device__ __forceinline__ void each_slot_of(F&& f, std::integer_sequence<int, P...>) {
    (f(Slot<P>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void each_slot(F&& f) {
    each_slot_of(f, std::make_integer_sequence<int, N>{});
}

// A 32-bit lane offset that the compiler widens beside the access (and not
// once, before the loop, into a register pair): a uniform base plus a 32-bit
// offset is an addressing mode of the global loads.
__device__ __forceinline__ std::uint32_t lane_offset(std::uint32_t& off) {
    asm volatile("" : "+v"(off));
    return off;
}
__device__ __forceinline__ std::uint64_t lane_offset(std::uint64_t& off) { return off; }

// Rows of at most this many columns keep every lane offset of a tile (up to
// 256 rows of fp16) below 2^32.
constexpr int kNarrowK = 1 << 22;

__device__ __forceinline__ std::uint32_t pack_half2(float a, float b) {
    return static_cast<std::uint32_t>(__half_as_ushort(from_f32<__half>(a))) |
           static_cast<std::uint32_t>(__half_as_ushort(from_f32<__half>(b))) << 16;
}

// Sums the WK partial tiles [WK][ROWS][P] (fp32, in LDS) in wave order and
// stores the fp16 rows in 16-byte units; token_of maps a tile row to its token.
template <int WK, int ROWS, int TN, int P, int T, class Token>
__device__ __forceinline__ void store_partials(const float* o_lds, __half* out, int tokens, int n, int n0,
                                               Token&& token_of) {
    const bool vec = (n % 8) == 0 && (reinterpret_cast<std::uintptr_t>(out) & 15) == 0;
    for (int u = threadIdx.x; u < ROWS * TN / 8; u += T) {
        const int row = u / (TN / 8), col = (u % (TN / 8)) * 8;
        const int t = token_of(row);
        if (t >= tokens || n0 + col >= n) continue;
        float v[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < WK; ++w) {
            const auto* src = reinterpret_cast<const float4*>(o_lds + (w * ROWS + row) * P + col);
            const float4 a = src[0], b = src[1];
            v[0] += a.x; v[1] += a.y; v[2] += a.z; v[3] += a.w;
            v[4] += b.x; v[5] += b.y; v[6] += b.z; v[7] += b.w;
        }
        __half* dst = out + static_cast<std::int64_t>(t) * n + n0 + col;
        if (vec) {
            *reinterpret_cast<uint4*>(dst) =
                make_uint4(pack_half2(v[0], v[1]), pack_half2(v[2], v[3]), pack_half2(v[4], v[5]), pack_half2(v[6], v[7]));
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (n0 + col + e < n) dst[e] = from_f32<__half>(v[e]);
        }
    }
}

}  // namespace
}  // namespace vt
