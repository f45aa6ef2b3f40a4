// W8A8 projection for many tokens on int8 matrix cores with a free fp32 order
// (the "mfma" A8 route above the decode kernels).
//
// out[t][n] = fp16( sum_p sum_g d[p][t][n][g] * ws[n][g] * as[p][t][g] )
//
// d is the exact integer dot of the group's 32 activation and weight codes
// (q8_dp4a.cuh:47-58), one v_mfma_i32_16x16x32_i8 on the codes as they are
// stored. The accumulator starts at the bit pattern of 1.5 * 2^23, so its 32
// bits read as a float are exactly 1.5 * 2^23 + d (|d| < 2^19) without a
// conversion, and one FMA with ws takes the offset off again:
//   t = fma(1.5 * 2^23 + d, ws, -1.5 * 2^23 * ws) = round(d * ws),
// because 1.5 * 2^23 * ws is exact (an 11-bit significand times 3); then
// y = fma(t, as, y). Two VALU instructions per output and group, as the
// reference's product and FMA (q8_dp4a.cuh:59-70), with one fp32 rounding
// besides the sum's as there. A wave sums its groups in the order it visits
// them (the passes' last, perhaps partial, stages or chunks first, then the
// others of each pass from column 0 up) and the sums of the waves that split K
// are added in wave order. The order depends on shape and tiling only: outputs
// are deterministic and agree with the reference to fp32 association, not bit
// for bit. The second pass of the residual profile is a second run over the
// same weight columns. (A row with a non-finite weight scale, which the format
// excludes, gives NaN.)
//
// Per 16 x 16 tile and group there are eight VALU instructions beside one MFMA
// of 16 cycles. So the two forms (cooperative and split, prefill.hpp) keep
// everything else off the VALU: codes go from memory through LDS into the MFMA
// unconverted, an operand is replaced by the next group's as soon as its last
// use is issued, and a tile's MFMA is issued four tiles before its VALU work.
// What binds it then is closest to the VALU, but not that alone. Counters,
// [34816 x 5120] at 2048 tokens: 10.1 VALU instructions per MFMA, VALU busy at
// most 69% of the time (4 cycles per instruction; an FMA measured 2.7 in a
// dense loop, which gives 46%), matrix cores 27%, LDS 20%, waves waiting 26% of
// theirs, two waves per SIMD. Measured on MI355X against the form this
// replaces (codes converted to fp16 once per workgroup, one 8-wave workgroup
// per 128- or 256-token tile, a barrier per group), us:
//   tokens x [7168 x 5120]: 64: 114 -> 18, 200: 119 -> 38, 512: 129 -> 66;
//   [5120 x 17408]: 64: 395 -> 54, 512: 422 -> 175;
//   [34816 x 5120], 2048 tokens: 1794 -> 1135 (643 TOP/s).
// At 100-128 tokens over 34816 rows of 64-512 columns, and at 1024 tokens over
// very many rows of up to 136, it is 1.12-1.20 times the time of the replaced
// form: prologue and output, not the K loop, are the time there.
#include "prefill.hpp"

#include <algorithm>

namespace vt {
namespace {

typedef int int4v __attribute__((ext_vector_type(4)));
typedef std::uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));  // a 16-byte load at 4-byte alignment

constexpr int kMagicBits = 0x4B400000;         // 1.5 * 2^23
constexpr float kMagic = 12582912.0f;

// A wave's TI x TJ tiles of 16 tokens x 16 rows. The MFMA's rows are weight
// rows and its columns tokens: lane (r, q) holds token r and rows 4q .. 4q + 3
// of a tile, its activation scale is one register per token tile and its
// weight scales four per row tile.
template <int TI, int TJ>
struct A8Tile {
    static constexpr int kTiles = TI * TJ, kAhead = kTiles < 5 ? 2 : 4;
    float4v y[TJ][TI];
    long fa[TI], fb[TJ];
    float as[TI];
    float4 ws[TJ];

    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int i = 0; i < TI; ++i) y[j][i] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // Reads all operands of a group.
    template <class Source>
    __device__ __forceinline__ void fill(const Source& src) {
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            fa[i] = src.a(i);
            as[i] = src.a_scale(i);
        }
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            fb[j] = src.b(j);
            ws[j] = src.b_scale(j);
        }
    }
    // Multiplies the group in registers and replaces every operand by the next
    // group's as soon as its last use is issued. Tiles run down the tokens of a
    // row tile; a tile's MFMA is issued kAhead tiles before its eight VALU
    // instructions. hook(t) runs before tile t.
    template <class Source, class Hook>
    __device__ __forceinline__ void group(const Source& next, Hook&& hook) {
        const int4v magic = {kMagicBits, kMagicBits, kMagicBits, kMagicBits};
        int4v d[kAhead];
        float4 nm;
#pragma unroll
        for (int t = 0; t < kTiles + kAhead; ++t) {
            hook(t);
            if (t >= kAhead) {
                const int f = t - kAhead, j = f / TI, i = f % TI;
                if (i == 0) nm = make_float4(-kMagic * ws[j].x, -kMagic * ws[j].y, -kMagic * ws[j].z, -kMagic * ws[j].w);
                const float s[4] = {ws[j].x, ws[j].y, ws[j].z, ws[j].w}, m[4] = {nm.x, nm.y, nm.z, nm.w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    y[j][i][e] = fmaf(fmaf(__int_as_float(d[f % kAhead][e]), s[e], m[e]), as[i], y[j][i][e]);
                if (j == TJ - 1) as[i] = next.a_scale(i);
                if (i == TI - 1) ws[j] = next.b_scale(j);
            }
            if (t < kTiles) {
                const int j = t / TI, i = t % TI;
                d[t % kAhead] = __builtin_amdgcn_mfma_i32_16x16x32_i8(fb[j], fa[i], magic, 0, 0, 0);
                if (j == TJ - 1) fa[i] = next.a(i);
                if (i == TI - 1) fb[j] = next.b(j);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // Partial sums of token tiles [I0, I0 + N) as fp32 rows of P floats.
    template <int I0, int N, int P>
    __device__ __forceinline__ void put(float* rows, int r, int q) const {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j)
                *reinterpret_cast<float4v*>(rows + (i * 16 + r) * P + j * 16 + 4 * q) = y[j][I0 + i];
    }
};

// Where a wave's operands of one group lie in LDS (byte addresses of its lane).
struct A8Source {
    const unsigned char *pa, *pb, *psa, *psb;
    int a_stride, b_stride;  // bytes between tiles of 16 rows
    __device__ __forceinline__ long a(int i) const { return *reinterpret_cast<const long*>(pa + i * a_stride); }
    __device__ __forceinline__ long b(int j) const { return *reinterpret_cast<const long*>(pb + j * b_stride); }
    __device__ __forceinline__ float a_scale(int i) const { return *reinterpret_cast<const float*>(psa + i * 64); }
    __device__ __forceinline__ float4 b_scale(int j) const { return *reinterpret_cast<const float4*>(psb + j * 64); }
};

template <int WT, int WN, int WK, int TI, int TJ>
struct A8Geom {
    static constexpr int kThreads = WT * WN * WK * 64;
    static constexpr int kTM = WT * TI * 16, kTN = WN * TJ * 16;
    static constexpr int kGroups = WK;      // groups per stage, one per K wave
    static constexpr int kU = 2 * kGroups;  // 16-byte units of a staged row of codes
    static constexpr int kAPer = (kTM * kU + kThreads - 1) / kThreads, kBPer = (kTN * kU + kThreads - 1) / kThreads;
    static constexpr int kAsPer = (kTM * kGroups + kThreads - 1) / kThreads;
    static constexpr int kWsPer = (kTN * kGroups + kThreads - 1) / kThreads;
    // A buffer holds whole rounds of the threads' stores, so no store is guarded.
    static constexpr int kB = kAPer * kThreads * 16, kAs = kB + kBPer * kThreads * 16, kWs = kAs + kAsPer * kThreads * 4;
    static constexpr int kStage = kWs + kWsPer * kThreads * 4;
    static constexpr int kPitch = kTN + 4;
    static constexpr int out_bytes(int oi) { return WK * WT * oi * 16 * kPitch * 4; }
    static constexpr int kOI = out_bytes(TI) <= 140 * 1024       ? TI
                               : TI % 2 == 0 && out_bytes(TI / 2) <= 140 * 1024 ? TI / 2
                               : TI % 4 == 0                                   ? TI / 4
                                                                               : 1;
    static constexpr int kLds = 2 * kStage > out_bytes(kOI) ? 2 * kStage : out_bytes(kOI);
    static_assert(TI % kOI == 0 && kLds <= 160 * 1024, "prefill tile exceeds LDS");
};

// Cooperative form: stages of WK groups in two LDS buffers, one group per K
// wave. While a stage is multiplied, the next one's operands are read, the one
// after is written to LDS and the one after that is requested.
template <int WT, int WN, int WK, int TI, int TJ, class Off>
__global__ __launch_bounds__(WT * WN * WK * 64, 2) void a8_prefill(const std::int8_t* __restrict__ acodes,
                                                                  const float* __restrict__ ascales,
                                                                  const std::int8_t* __restrict__ wcodes,
                                                                  const __half* __restrict__ wscales,
                                                                  __half* __restrict__ out, int tokens, int n,
                                                                  int padded, int groups, int passes, TileOrder order) {
    using G = A8Geom<WT, WN, WK, TI, TJ>;
    constexpr int TM = G::kTM, TN = G::kTN, T = G::kThreads, U = G::kU, KG = G::kGroups;
    extern __shared__ uint4 a8p_lds[];
    auto* lds = reinterpret_cast<unsigned char*>(a8p_lds);
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wn = (wave / WK) % WN, wt = wave / (WK * WN);
    const int q = lane >> 4, r = lane & 15;
    const int tile = tile_of(order);
    if (tile < 0) return;
    const int t0 = tile % order.token_tiles * TM, n0 = tile / order.token_tiles * TN;

    const std::int64_t count = static_cast<std::int64_t>(tokens) * groups;  // groups of one pass
    const auto* a_base = reinterpret_cast<const char*>(acodes) + static_cast<std::int64_t>(t0) * groups * 32;
    const auto* as_base = reinterpret_cast<const char*>(ascales + static_cast<std::int64_t>(t0) * groups);
    const auto* b_base = reinterpret_cast<const char*>(wcodes + static_cast<std::int64_t>(n0) * padded);
    const auto* ws_base = reinterpret_cast<const char*>(wscales + static_cast<std::int64_t>(n0) * (padded / 32));
    Off a_off[G::kAPer], b_off[G::kBPer], as_off[G::kAsPer], ws_off[G::kWsPer];
    std::uint32_t a_put[G::kAPer], b_put[G::kBPer], as_put[G::kAsPer], ws_put[G::kWsPer];
#pragma unroll
    for (int u = 0; u < G::kAPer; ++u) {
        const int i = tid + u * T, row = i / U;
        a_off[u] = static_cast<Off>(min(row, tokens - 1 - t0)) * (groups * 32) + 16 * (i % U);
        a_put[u] = 16 * (row * U + ((i % U) ^ swizzle<U>(row)));
    }
#pragma unroll
    for (int u = 0; u < G::kBPer; ++u) {
        const int i = tid + u * T, row = i / U;
        b_off[u] = static_cast<Off>(min(row, n - 1 - n0)) * padded + 16 * (i % U);
        b_put[u] = G::kB + 16 * (row * U + ((i % U) ^ swizzle<U>(row)));
    }
#pragma unroll
    for (int u = 0; u < G::kAsPer; ++u) {
        const int i = tid + u * T;
        as_off[u] = 4u * (static_cast<Off>(min(i / KG, tokens - 1 - t0)) * groups + i % KG);
        as_put[u] = G::kAs + 4 * (i < TM * KG ? (i % KG) * TM + i / KG : i);
    }
#pragma unroll
    for (int u = 0; u < G::kWsPer; ++u) {
        const int i = tid + u * T;
        ws_off[u] = 2u * (static_cast<Off>(min(i / KG, n - 1 - n0)) * (padded / 32) + i % KG);
        ws_put[u] = G::kWs + 4 * (i < TN * KG ? (i % KG) * TN + i / KG : i);
    }

    // Stage order: the partial stage of each pass first (when the groups are
    // not whole stages), so that only the prologue clamps, then the whole
    // stages of pass 0 and of pass 1.
    const int whole = groups / KG, edges = whole * KG < groups ? passes : 0;
    const int stages = edges + passes * whole;
    struct Stage {
        u32x4 a[G::kAPer], b[G::kBPer];
        float as[G::kAsPer];
        unsigned short ws[G::kWsPer];
    };
    Stage st;
    auto load = [&](int stage, Stage& st) __attribute__((always_inline)) {
        const int w = min(max(stage - edges, 0), max(passes * whole - 1, 0));
        const int pass = w >= whole && w > 0 ? 1 : 0;
        const std::int64_t base = w - pass * whole;
        const char* ap = a_base + pass * count * 32 + base * (32 * KG);
        const char* sp = as_base + pass * count * 4 + base * (4 * KG);
        const char* bp = b_base + base * (32 * KG);
        const char* wp = ws_base + base * (2 * KG);
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u) st.a[u] = *reinterpret_cast<const u32x4*>(ap + lane_offset(a_off[u]));
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u) st.b[u] = *reinterpret_cast<const u32x4*>(bp + lane_offset(b_off[u]));
#pragma unroll
        for (int u = 0; u < G::kAsPer; ++u) st.as[u] = *reinterpret_cast<const float*>(sp + lane_offset(as_off[u]));
#pragma unroll
        for (int u = 0; u < G::kWsPer; ++u)
            st.ws[u] = *reinterpret_cast<const unsigned short*>(wp + lane_offset(ws_off[u]));
    };
    // The partial stage of a pass: groups past the last one carry scale 0 (their codes are clamped, finite).
    auto load_edge = [&](int pass, Stage& st) __attribute__((always_inline)) {
        const int g0 = whole * KG;
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u) {
            const int unit = (tid + u * T) % U;
            st.a[u] = *reinterpret_cast<const u32x4*>(
                a_base + pass * count * 32 + a_off[u] + 16 * static_cast<std::int64_t>(min(2 * g0, 2 * groups - 1 - unit)));
        }
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u) {
            const int unit = (tid + u * T) % U;
            st.b[u] = *reinterpret_cast<const u32x4*>(
                b_base + b_off[u] + 16 * static_cast<std::int64_t>(min(2 * g0, 2 * groups - 1 - unit)));
        }
#pragma unroll
        for (int u = 0; u < G::kAsPer; ++u) {
            const int g = (tid + u * T) % KG;
            const float v = *reinterpret_cast<const float*>(as_base + pass * count * 4 + as_off[u] +
                                                            4 * static_cast<std::int64_t>(min(g0, groups - 1 - g)));
            st.as[u] = g0 + g < groups ? v : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < G::kWsPer; ++u) {
            const int g = (tid + u * T) % KG;
            const unsigned short v = *reinterpret_cast<const unsigned short*>(
                ws_base + ws_off[u] + 2 * static_cast<std::int64_t>(min(g0, groups - 1 - g)));
            st.ws[u] = g0 + g < groups ? v : 0;
        }
    };
    auto store = [&](int buf, const Stage& st) __attribute__((always_inline)) {
        unsigned char* base = lds + buf * G::kStage;
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u) *reinterpret_cast<u32x4*>(base + a_put[u]) = st.a[u];
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u) *reinterpret_cast<u32x4*>(base + b_put[u]) = st.b[u];
#pragma unroll
        for (int u = 0; u < G::kAsPer; ++u) *reinterpret_cast<float*>(base + as_put[u]) = st.as[u];
#pragma unroll
        for (int u = 0; u < G::kWsPer; ++u)
            *reinterpret_cast<float*>(base + ws_put[u]) = __half2float(__ushort_as_half(st.ws[u]));
    };
    const std::uint32_t a_get = 16 * ((wt * TI * 16 + r) * U + ((2 * wk + (q >> 1)) ^ swizzle<U>(r))) + 8 * (q & 1);
    const std::uint32_t b_get =
        G::kB + 16 * ((wn * TJ * 16 + r) * U + ((2 * wk + (q >> 1)) ^ swizzle<U>(r))) + 8 * (q & 1);
    const std::uint32_t as_get = G::kAs + 4 * (wk * TM + wt * TI * 16 + r);
    const std::uint32_t ws_get = G::kWs + 4 * (wk * TN + wn * TJ * 16 + 4 * q);
    auto source = [&](int buf) __attribute__((always_inline)) {
        const unsigned char* base = lds + buf * G::kStage;
        return A8Source{base + a_get, base + b_get, base + as_get, base + ws_get, 256 * U, 256 * U};
    };

    A8Tile<TI, TJ> m;
    m.clear();
    {  // the first two stages are requested together: for short rows the prologue is most of the time
        Stage first;
        if (edges > 0) load_edge(0, first);
        else load(0, first);
        if (edges > 1) load_edge(1, st);
        else if (stages > 1) load(1, st);
        store(0, first);
        if (stages > 1) store(1, st);
    }
    if (whole == 0) {  // no whole stage: the loop's requests (never consumed) stay on group 0 of their rows
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u) a_off[u] -= 16 * ((tid + u * T) % U);
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u) b_off[u] -= 16 * ((tid + u * T) % U);
#pragma unroll
        for (int u = 0; u < G::kAsPer; ++u) as_off[u] -= 4 * ((tid + u * T) % KG);
#pragma unroll
        for (int u = 0; u < G::kWsPer; ++u) ws_off[u] -= 2 * ((tid + u * T) % KG);
    }
    load(2, st);
    __syncthreads();
    m.fill(source(0));
    __syncthreads();
    constexpr int kStoreAt = TI * TJ / 4, kLoadAt = TI * TJ / 4 + 2;
    for (int sg = 0; sg < stages; ++sg) {
        m.group(source((sg + 1) & 1), [&](int t) __attribute__((always_inline)) {
            if (t == kStoreAt) store(sg & 1, st);
            if (t == kLoadAt) load(sg + 3, st);
        });
        __syncthreads();
    }

    auto* o_lds = reinterpret_cast<float*>(lds);
    constexpr int OI = G::kOI, P = G::kPitch, kRows = WT * OI * 16;
    each_slot<TI / OI>([&](auto c) __attribute__((always_inline)) {
        __syncthreads();
        m.template put<c * OI, OI, P>(o_lds + (wk * kRows + wt * OI * 16) * P + wn * TJ * 16, r, q);
        __syncthreads();
        store_partials<WK, kRows, TN, P, T>(o_lds, out, tokens, n, n0, [&](int row) {
            return t0 + (row / (OI * 16)) * TI * 16 + c * OI * 16 + row % (OI * 16);
        });
    });
}

template <int WK, int TI, int TJ>
struct A8SplitGeom {
    static constexpr int kThreads = WK * 64;
    static constexpr int kTM = TI * 16, kTN = TJ * 16;
    static constexpr int kAsPer = (kTM + 63) / 64;
    static constexpr int kB = kTM * 128, kAs = kB + kTN * 128, kWs = kAs + 4 * kAsPer * 64 * 4;
    static constexpr int kWave = kWs + 4 * 64 * 4;
    static constexpr int kPitch = kTN + 4;
    static constexpr int kOut = WK * kTM * kPitch * 4;
    static constexpr int kLds = WK * kWave > kOut ? WK * kWave : kOut;
    static_assert(kTN <= 64 && kLds <= 160 * 1024, "split tile exceeds LDS");
};

// Split form: every wave computes the whole tile over its own 128-column
// chunks through its own LDS region (a wave's LDS accesses stay in order), so
// there is no barrier before the final sum.
template <int WK, int TI, int TJ>
__global__ __launch_bounds__(WK * 64, 2) void a8_prefill_split(const std::int8_t* __restrict__ acodes,
                                                              const float* __restrict__ ascales,
                                                              const std::int8_t* __restrict__ wcodes,
                                                              const __half* __restrict__ wscales,
                                                              __half* __restrict__ out, int tokens, int n, int padded,
                                                              int groups, int passes, TileOrder order) {
    using G = A8SplitGeom<WK, TI, TJ>;
    constexpr int TM = G::kTM, TN = G::kTN, kA = 2 * TI, kB = 2 * TJ;
    static_assert(WK >= 2, "the last chunk of each pass is a wave's first");
    extern __shared__ uint4 a8p_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, r = lane & 15;
    const int tile = tile_of(order);
    if (tile < 0) return;
    const int t0 = tile % order.token_tiles * TM, n0 = tile / order.token_tiles * TN;
    auto* lds = reinterpret_cast<unsigned char*>(a8p_lds) + wave * G::kWave;

    // Chunk order: the last chunk of each pass (it may be partial) first, then
    // the others of pass 0 and of pass 1; wave w takes every WK-th from w.
    const int chunks = padded / 128, inner = chunks - 1, total = passes * chunks;
    A8Tile<TI, TJ> m;
    m.clear();
    if (wave < total) {
        const std::int64_t count = static_cast<std::int64_t>(tokens) * groups;
        const auto* a_base = reinterpret_cast<const char*>(acodes) + static_cast<std::int64_t>(t0) * groups * 32;
        const auto* as_base = reinterpret_cast<const char*>(ascales + static_cast<std::int64_t>(t0) * groups);
        const auto* b_base = reinterpret_cast<const char*>(wcodes + static_cast<std::int64_t>(n0) * padded);
        const auto* ws_base = reinterpret_cast<const char*>(wscales + static_cast<std::int64_t>(n0) * (padded / 32));
        // Code unit u of a lane: row lane / 8 + 8 u, unit lane % 8 of its 128 bytes.
        std::uint32_t a_off[kA], b_off[kB], as_off[G::kAsPer], ws_off;
#pragma unroll
        for (int u = 0; u < kA; ++u)
            a_off[u] = static_cast<std::uint32_t>(min(lane / 8 + 8 * u, tokens - 1 - t0)) * (groups * 32) + 16 * (lane % 8);
#pragma unroll
        for (int u = 0; u < kB; ++u)
            b_off[u] = static_cast<std::uint32_t>(min(lane / 8 + 8 * u, n - 1 - n0)) * padded + 16 * (lane % 8);
#pragma unroll
        for (int u = 0; u < G::kAsPer; ++u)
            as_off[u] = 4u * static_cast<std::uint32_t>(min(lane + 64 * u, tokens - 1 - t0)) * groups;
        ws_off = 2u * static_cast<std::uint32_t>(min(lane, n - 1 - n0)) * (padded / 32);
        u32x4 st_a[kA], st_b[kB];
        float4u st_as[G::kAsPer];
        uint2 st_ws;
        // A chunk of four whole groups (inner chunks; past the end, chunk 0 of pass 0, never consumed).
        auto load = [&](int v) __attribute__((always_inline)) {
            const int w = v < total ? v - passes : 0;
            const int pass = w >= inner && w > 0 ? 1 : 0;
            const std::int64_t c = w - pass * inner;
            const char* ap = a_base + pass * count * 32 + c * 128;
            const char* sp = as_base + pass * count * 4 + c * 16;
#pragma unroll
            for (int u = 0; u < kA; ++u) st_a[u] = *reinterpret_cast<const u32x4*>(ap + lane_offset(a_off[u]));
#pragma unroll
            for (int u = 0; u < kB; ++u) st_b[u] = *reinterpret_cast<const u32x4*>(b_base + c * 128 + lane_offset(b_off[u]));
#pragma unroll
            for (int u = 0; u < G::kAsPer; ++u) st_as[u] = *reinterpret_cast<const float4u*>(sp + lane_offset(as_off[u]));
            st_ws = *reinterpret_cast<const uint2*>(ws_base + c * 8 + lane_offset(ws_off));
        };
        // The last chunk of a pass: groups past the last one carry scale 0 (their codes are clamped, finite).
        auto load_edge = [&](int pass) __attribute__((always_inline)) {
            const int real = groups - 4 * inner;  // 1 .. 4
            const int unit = min(8 * inner, 2 * groups - 1 - lane % 8);
#pragma unroll
            for (int u = 0; u < kA; ++u)
                st_a[u] = *reinterpret_cast<const u32x4*>(a_base + pass * count * 32 + a_off[u] + 16 * static_cast<std::int64_t>(unit));
#pragma unroll
            for (int u = 0; u < kB; ++u)
                st_b[u] = *reinterpret_cast<const u32x4*>(b_base + b_off[u] + 16 * static_cast<std::int64_t>(unit));
#pragma unroll
            for (int u = 0; u < G::kAsPer; ++u)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float v = *reinterpret_cast<const float*>(
                        as_base + pass * count * 4 + as_off[u] + 4 * static_cast<std::int64_t>(min(4 * inner + g, groups - 1)));
                    st_as[u][g] = g < real ? v : 0.0f;
                }
            const uint2 v = *reinterpret_cast<const uint2*>(ws_base + ws_off + 8 * static_cast<std::int64_t>(inner));
            st_ws.x = real >= 2 ? v.x : v.x & 0xffffu;
            st_ws.y = real >= 4 ? v.y : real == 3 ? v.y & 0xffffu : 0u;
        };
        // Rows 8 apart alternate between two swizzles.
        std::uint32_t put[2];
#pragma unroll
        for (int odd = 0; odd < 2; ++odd) put[odd] = 16 * ((lane / 8) * 8 + ((lane % 8) ^ swizzle<8>(lane / 8 + 8 * odd)));
        auto store = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int u = 0; u < kA; ++u) *reinterpret_cast<u32x4*>(lds + put[u & 1] + u * 1024) = st_a[u];
#pragma unroll
            for (int u = 0; u < kB; ++u) *reinterpret_cast<u32x4*>(lds + G::kB + put[u & 1] + u * 1024) = st_b[u];
#pragma unroll
            for (int u = 0; u < G::kAsPer; ++u)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<float*>(lds + G::kAs + 4 * ((g * G::kAsPer + u) * 64 + lane)) = st_as[u][g];
            const float f[4] = {half_lo(st_ws.x), half_hi(st_ws.x), half_lo(st_ws.y), half_hi(st_ws.y)};
#pragma unroll
            for (int g = 0; g < 4; ++g) *reinterpret_cast<float*>(lds + G::kWs + 4 * (64 * g + lane)) = f[g];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        };
        std::uint32_t get[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) get[g] = 16 * (r * 8 + ((2 * g + (q >> 1)) ^ swizzle<8>(r))) + 8 * (q & 1);
        auto source = [&](int g) __attribute__((always_inline)) {
            return A8Source{lds + get[g], lds + G::kB + get[g], lds + G::kAs + 4 * (g * G::kAsPer * 64 + r),
                            lds + G::kWs + 4 * (64 * g + 4 * q), 2048, 2048};
        };
        if (wave < passes) {
            load_edge(wave);
            store();
        } else {
            load(wave);
            store();
        }
        load(wave + WK);
        m.fill(source(0));
        for (int v = wave; v < total; v += WK) {
            each_slot<4>([&](auto g) __attribute__((always_inline)) {
                m.group(source((g + 1) % 4), [&](int t) __attribute__((always_inline)) {
                    if (g == 3 && t == 0) {  // every read of this chunk is issued
                        store();
                        load(v + 2 * WK);
                    }
                });
            });
        }
    }

    auto* o_lds = reinterpret_cast<float*>(a8p_lds);
    constexpr int P = G::kPitch;
    __syncthreads();
    m.template put<0, TI, P>(o_lds + wave * TM * P, r, q);
    __syncthreads();
    store_partials<WK, TM, TN, P, G::kThreads>(o_lds, out, tokens, n, n0, [&](int row) { return t0 + row; });
}

// The split form over the tiled Q8 planes (the decode route's copy: codes
// [row block][64-column chunk][lane 16q + m][two groups' 8 bytes], scales
// [row block][chunk][row][2]), for 17-32 tokens, and for fewer whose
// activations exceed the decode kernels' LDS outside 513-768 row blocks. A lane's 16 code bytes are its
// fragments of a chunk's two groups and its 16 scale bytes the four rows'
// pairs, so weights go straight to registers in 1 KB wave loads; activations
// travel through the wave's LDS region as in the row-major form.
template <int WK, int TI, int TJ>
struct A8TiledGeom {
    static constexpr int kThreads = WK * 64;
    static constexpr int kTM = TI * 16, kTN = TJ * 16;
    static constexpr int kAs = kTM * 128, kWave = kAs + 4 * 64 * 4;
    static constexpr int kPitch = kTN + 4;
    static constexpr int kOut = WK * kTM * kPitch * 4;
    static constexpr int kLds = WK * kWave > kOut ? WK * kWave : kOut;
    static_assert(kTM <= 64 && kLds <= 64 * 1024, "tiled split tile exceeds the default LDS limit");
};

template <int TJ>
struct A8TiledSource {
    const unsigned char *pa, *psa;
    const u32x4 *codes, *scales;  // [TJ] of the 64-column chunk that holds the group
    int odd;                      // second group of the chunk
    __device__ __forceinline__ long a(int i) const { return *reinterpret_cast<const long*>(pa + i * 2048); }
    __device__ __forceinline__ float a_scale(int i) const { return *reinterpret_cast<const float*>(psa + i * 64); }
    __device__ __forceinline__ long b(int j) const {
        return static_cast<long>(static_cast<std::uint64_t>(codes[j][2 * odd]) |
                                 static_cast<std::uint64_t>(codes[j][2 * odd + 1]) << 32);
    }
    __device__ __forceinline__ float4 b_scale(int j) const {
        const u32x4 s = scales[j];
        return odd ? make_float4(half_hi(s[0]), half_hi(s[1]), half_hi(s[2]), half_hi(s[3]))
                   : make_float4(half_lo(s[0]), half_lo(s[1]), half_lo(s[2]), half_lo(s[3]));
    }
};

template <int WK, int TI, int TJ>
__global__ __launch_bounds__(WK * 64, WK > 8 ? WK / 4 : 2) void a8_tiled_split(
    const std::int8_t* __restrict__ acodes, const float* __restrict__ ascales, const u32x4* __restrict__ wcodes,
    const u32x4* __restrict__ wscales, __half* __restrict__ out, int tokens, int n, int padded, int groups, int passes) {
    using G = A8TiledGeom<WK, TI, TJ>;
    constexpr int TM = G::kTM, TN = G::kTN, kA = 2 * TI;
    static_assert(WK >= 2, "the last chunk of each pass is a wave's first");
    extern __shared__ uint4 a8p_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, r = lane & 15;
    const int block0 = blockIdx.x * TJ, blocks = (n + 15) / 16;
    auto* lds = reinterpret_cast<unsigned char*>(a8p_lds) + wave * G::kWave;

    const int chunks = padded / 128, inner = chunks - 1, total = passes * chunks;
    A8Tile<TI, TJ> m;
    m.clear();
    if (wave < total) {
        const std::int64_t count = static_cast<std::int64_t>(tokens) * groups;
        // Activation unit u of a lane: row lane / 8 + 8 u, unit lane % 8 of the
        // chunk's 128 bytes; scales: row lane. Where the only chunk is partial,
        // the requests that are never consumed stay inside the first row.
        const std::int8_t* a_src[kA];
        const bool whole = inner > 0 || groups >= 4;
#pragma unroll
        for (int u = 0; u < kA; ++u)
            a_src[u] = acodes + static_cast<std::int64_t>(min(lane / 8 + 8 * u, tokens - 1)) * groups * 32 +
                       (whole ? 16 * (lane % 8) : 0);
        const float* as_src = ascales + (whole ? static_cast<std::int64_t>(min(lane, tokens - 1)) * groups : 0);
        const u32x4 *b_src[TJ], *s_src[TJ];
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const std::int64_t blk = min(block0 + j, blocks - 1);  // clamped blocks are never stored
            b_src[j] = wcodes + blk * (2 * chunks) * 64 + lane;
            s_src[j] = wscales + blk * (2 * chunks) * 4 + q;
        }
        u32x4 st_a[kA], codes[2][TJ], scales[2][TJ];
        float4u st_as;
        // Virtual chunk v: the last chunk of each pass first, then the others;
        // past the end, chunk 0 of pass 0 (never consumed).
        auto locate = [&](int v, int& pass, std::int64_t& c) __attribute__((always_inline)) {
            const int w = v < total ? v - passes : 0;
            pass = v < passes ? v : w >= inner && w > 0 ? 1 : 0;
            c = v < passes ? inner : w - (w >= inner && w > 0 ? inner : 0);
        };
        auto load_b = [&](int v, int h) __attribute__((always_inline)) {
            int pass;
            std::int64_t c;
            locate(v, pass, c);
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                codes[h][j] = __builtin_nontemporal_load(b_src[j] + (2 * c + h) * 64);
                scales[h][j] = __builtin_nontemporal_load(s_src[j] + (2 * c + h) * 4);
            }
        };
        auto load_a = [&](int v) __attribute__((always_inline)) {
            int pass;
            std::int64_t c;
            locate(v, pass, c);
#pragma unroll
            for (int u = 0; u < kA; ++u)
                st_a[u] = *reinterpret_cast<const u32x4*>(a_src[u] + pass * count * 32 + c * 128);
            st_as = *reinterpret_cast<const float4u*>(as_src + pass * count + c * 4);
        };
        // The last chunk of a pass: groups past the last one carry scale 0 (their codes are clamped, finite).
        auto load_edge = [&](int pass) __attribute__((always_inline)) {
            const int real = groups - 4 * inner;  // 1 .. 4
            const int unit = min(8 * inner + lane % 8, 2 * groups - 1);
#pragma unroll
            for (int u = 0; u < kA; ++u)
                st_a[u] = *reinterpret_cast<const u32x4*>(
                    acodes + pass * count * 32 +
                    (static_cast<std::int64_t>(min(lane / 8 + 8 * u, tokens - 1)) * groups * 2 + unit) * 16);
            const float* as = ascales + pass * count + static_cast<std::int64_t>(min(lane, tokens - 1)) * groups;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float v = as[min(4 * inner + g, groups - 1)];
                st_as[g] = g < real ? v : 0.0f;
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < TJ; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const std::uint32_t keep = (2 * h < real ? 0x0000ffffu : 0u) | (2 * h + 1 < real ? 0xffff0000u : 0u);
                        scales[h][j][e] &= keep;
                    }
        };
        std::uint32_t put[2];
#pragma unroll
        for (int odd = 0; odd < 2; ++odd) put[odd] = 16 * ((lane / 8) * 8 + ((lane % 8) ^ swizzle<8>(lane / 8 + 8 * odd)));
        auto store = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int u = 0; u < kA; ++u) *reinterpret_cast<u32x4*>(lds + put[u & 1] + u * 1024) = st_a[u];
#pragma unroll
            for (int g = 0; g < 4; ++g) *reinterpret_cast<float*>(lds + G::kAs + 4 * (64 * g + lane)) = st_as[g];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        };
        std::uint32_t get[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) get[g] = 16 * (r * 8 + ((2 * g + (q >> 1)) ^ swizzle<8>(r))) + 8 * (q & 1);
        auto source = [&](auto g) __attribute__((always_inline)) {
            return A8TiledSource<TJ>{lds + get[g], lds + G::kAs + 4 * (64 * g + r), codes[g / 2], scales[g / 2], g % 2};
        };
        load_b(wave, 0);
        load_b(wave, 1);
        if (wave < passes) {
            load_edge(wave);
            store();
        } else {
            load_a(wave);
            store();
        }
        load_a(wave + WK);
        m.fill(source(Slot<0>{}));
        for (int v = wave; v < total; v += WK) {
            each_slot<4>([&](auto g) __attribute__((always_inline)) {
                m.group(source(Slot<(g + 1) % 4>{}), [&](int t) __attribute__((always_inline)) {
                    // The first half of the chunk is in use until group 1's
                    // operands are taken, the second until group 3's.
                    if (g == 1 && t == 0) load_b(v + WK, 0);
                    if (g == 3 && t == 0) {
                        load_b(v + WK, 1);
                        store();  // every read of this chunk is issued
                        load_a(v + 2 * WK);
                    }
                });
            });
        }
    }

    auto* o_lds = reinterpret_cast<float*>(a8p_lds);
    constexpr int P = G::kPitch;
    __syncthreads();
    m.template put<0, TI, P>(o_lds + wave * TM * P, r, q);
    __syncthreads();
    store_partials<WK, TM, TN, P, G::kThreads>(o_lds, out, tokens, n, block0 * 16, [&](int row) { return row; });
}

struct A8Operands {
    const std::int8_t* acodes;
    const float* ascales;
    const std::int8_t* codes;
    const __half* scales;
    __half* out;
    int tokens, n, padded, groups, passes;
};

template <int WT, int WN, int WK, int TI, int TJ, class Off = std::uint32_t>
void launch_coop(const A8Operands& o, hipStream_t stream) {
    using G = A8Geom<WT, WN, WK, TI, TJ>;
    const auto kernel = a8_prefill<WT, WN, WK, TI, TJ, Off>;
    const TileOrder order = tile_order(o.tokens, G::kTM, o.n, G::kTN);
    static LdsLimit limit;
    limit.raise(kernel, G::kLds);
    kernel<<<8 * order.per_xcd, G::kThreads, G::kLds, stream>>>(o.acodes, o.ascales, o.codes, o.scales, o.out, o.tokens,
                                                               o.n, o.padded, o.groups, o.passes, order);
}

template <int WK, int TI, int TJ>
void launch_split(const A8Operands& o, hipStream_t stream) {
    using G = A8SplitGeom<WK, TI, TJ>;
    const auto kernel = a8_prefill_split<WK, TI, TJ>;
    const TileOrder order = tile_order(o.tokens, G::kTM, o.n, G::kTN);
    static LdsLimit limit;
    limit.raise(kernel, G::kLds);
    kernel<<<8 * order.per_xcd, G::kThreads, G::kLds, stream>>>(o.acodes, o.ascales, o.codes, o.scales, o.out, o.tokens,
                                                               o.n, o.padded, o.groups, o.passes, order);
}

}  // namespace

void a8_fast_launch(const void* workspace, const std::int8_t* codes, const __half* scales, void* out, int tokens, int n,
                    int k, int padded, int passes, hipStream_t stream) {
    A8Operands o{};
    o.tokens = tokens; o.n = n; o.padded = padded; o.groups = (k + 31) / 32; o.passes = passes;
    const std::int64_t count = static_cast<std::int64_t>(tokens) * o.groups;
    o.acodes = static_cast<const std::int8_t*>(workspace);
    o.ascales = reinterpret_cast<const float*>(o.acodes + count * 32 * passes);
    o.codes = codes; o.scales = scales; o.out = static_cast<__half*>(out);
    if (k > kNarrowK) {  // rows too long for 32-bit lane offsets
        launch_coop<1, 2, 4, 4, 4, std::uint64_t>(o, stream);
        return;
    }
    // The tiling with the least predicted time (the passes run one after the
    // other over K); the constants are a fit to 770 shapes (33-8192
    // tokens, 256-151936 rows, 64-25600 columns; each candidate timed on each
    // shape on MI355X): the choice is within 11% of the fastest candidate on
    // every one of them and 0.2% on average. The three without a K split share
    // a CU (two or four workgroups) and win where K is short, so that prologue
    // and output count (16384 rows x 256 columns, 8192 tokens: 256 x 128 tiles
    // 228 us, these 184; 100 tokens x 34816 rows x 136: the fastest of the
    // others 16.2, these 9.0).
    constexpr PrefillTiling kTilings[12] = {
        {256, 128, 1, 1.1, 6.25, 24.46, 24.46}, {128, 128, 1, 0.0, 5.10, 12.71, 12.71}, {64, 128, 1, 0.7, 3.98, 7.14, 7.14},
        {128, 128, 2, 2.4, 2.96, 17.78, 30.71}, {64, 128, 4, 0.8, 1.64, 16.16, 54.83},  {32, 128, 4, 0.2, 0.00, 30.22, 68.00},
        {64, 64, 1, 1.7, 4.73, 3.48, 3.48},     {64, 64, 2, 1.8, 3.36, 4.10, 6.94},     {48, 64, 2, 1.9, 2.83, 3.60, 6.05},
        {48, 64, 1, 0.9, 4.41, 3.13, 3.13},     {32, 64, 1, 1.0, 2.96, 3.00, 3.00},     {32, 32, 1, 1.8, 0.88, 2.03, 2.03}};
    int best = fastest_tiling(kTilings, tokens, n, static_cast<double>(k) * passes);
    // The split form reads a chunk's four weight scales as one 8-byte word and
    // needs one whole chunk.
    if (best >= 6 && (k < 128 || !aligned(scales, 8))) best = k < 128 ? 4 : 2;
    switch (best) {
        case 0: launch_coop<2, 2, 2, 8, 4>(o, stream); break;
        case 1: launch_coop<1, 2, 4, 8, 4>(o, stream); break;
        case 2: launch_coop<1, 2, 4, 4, 4>(o, stream); break;
        case 3: launch_coop<1, 4, 1, 8, 2>(o, stream); break;
        case 4: launch_coop<1, 4, 1, 4, 2>(o, stream); break;
        case 5: launch_coop<1, 4, 1, 2, 2>(o, stream); break;
        case 6: launch_split<8, 4, 4>(o, stream); break;
        case 7: launch_split<4, 4, 4>(o, stream); break;
        case 8: launch_split<4, 3, 4>(o, stream); break;
        case 9: launch_split<8, 3, 4>(o, stream); break;
        case 10: launch_split<8, 2, 4>(o, stream); break;
        default: launch_split<8, 2, 2>(o, stream); break;
    }
}

template <int WK, int TI, int TJ>
void launch_tiled_split(const std::int8_t* acodes, const float* ascales, const u32x4* codes, const u32x4* scales,
                        __half* out, int tokens, int n, int padded, int groups, int passes, hipStream_t stream) {
    using G = A8TiledGeom<WK, TI, TJ>;
    a8_tiled_split<WK, TI, TJ><<<(n + G::kTN - 1) / G::kTN, G::kThreads, G::kLds, stream>>>(
        acodes, ascales, codes, scales, out, tokens, n, padded, groups, passes);
}

// Operands are admitted by the caller (a8_tiled_launch); at most 32 tokens.
void a8_tiled_split_launch(const void* workspace, const void* codes, const void* scales, void* out, int tokens, int n,
                           int k, int padded, int passes, hipStream_t stream) {
    const int groups = (k + 31) / 32;
    const std::int64_t count = static_cast<std::int64_t>(tokens) * groups;
    const auto* acodes = static_cast<const std::int8_t*>(workspace);
    const auto* ascales = reinterpret_cast<const float*>(acodes + count * 32 * passes);
    const auto* cp = static_cast<const u32x4*>(codes);
    const auto* sp = static_cast<const u32x4*>(scales);
    auto* op = static_cast<__half*>(out);
    const int blocks = (n + 15) / 16;
    auto launch = [&](auto waves, auto token_blocks, auto row_blocks) {
        launch_tiled_split<waves, token_blocks, row_blocks>(acodes, ascales, cp, sp, op, tokens, n, padded, groups, passes,
                                                            stream);
    };
    // Row blocks per workgroup so that up to 768 blocks make at most one
    // workgroup of eight K waves per CU; beyond, four K waves and two
    // workgroups per CU (at up to 16 tokens past 1024 blocks). MI355X, 32
    // tokens, one pass, against the per-lane fragment form this replaces, us:
    // 4096 x 4096 19.2 -> 8.5, 7168 x 5120 24.1 -> 15.2, 5120 x 17408 71 -> 35,
    // 11702 x 15232 106 -> 43, 34816 x 5120 106 -> 45; the neighbouring shapes
    // of the rule measured up to 1.5x slower there.
    if (tokens > 16) {
        if (blocks <= 256) launch(Slot<8>{}, Slot<2>{}, Slot<1>{});
        else if (blocks <= 512) launch(Slot<8>{}, Slot<2>{}, Slot<2>{});
        else if (blocks <= 768) launch(Slot<8>{}, Slot<2>{}, Slot<3>{});
        else launch(Slot<4>{}, Slot<2>{}, Slot<3>{});
    } else if (blocks <= 256) {
        launch(Slot<8>{}, Slot<1>{}, Slot<1>{});
    } else if (blocks <= 1024) {  // 513-768 blocks stay with the decode kernels
        launch(Slot<8>{}, Slot<1>{}, Slot<2>{});
    } else {
        launch(Slot<4>{}, Slot<1>{}, Slot<3>{});
    }
}

}  // namespace vt
