// Q4 W4A16 projection for many tokens (prefill, from 32 tokens) on fp16 matrix
// cores: the contract weights w = fp16(q * scale) (flash_next_q4.cu:7-14,
// weight_dequant.cuh:16-51), fp32 accumulation.
//
// Once the weights are fp16 the product is a plain fp16 GEMM, so no per-group
// work remains on the sums; what is left for the VALU is the dequantization,
// 16 instructions per 8 codes. Every wave dequantizes the fragments it
// multiplies (its 64 rows serve 16 TI tokens), so codes travel through LDS as
// 4 bits. Cooperative and split forms, tile order and tiling choice as in
// prefill.hpp; the activation fragments are replaced in place and the next
// slice's weights are dequantized beside the MFMAs of the current one.
//
// What binds it at these token counts: no unit alone. Counters, [5120 x 25600]
// at 128 tokens: 7.2 VALU instructions per MFMA (the dequantization per wave),
// VALU busy at most 41% of the time, matrix cores 23%, LDS 34% (320 bytes read
// per MFMA at 128 x 64 wave tiles; waves wait for it 14% of theirs), any wait
// 34%; one 64-column step of activations is in flight per wave. The 256-token
// tiles of row_prefill, whose workgroup dequantizes a weight once, stay the
// faster form from about 1000 tokens on. Measured on MI355X against row_prefill
// at every token count (grids of 128- and 256-token tiles, K serial), us:
//   tokens x [7168 x 5120]: 64: 56 -> 15.4, 200: 56 -> 32, 512: 107 -> 49;
//   [5120 x 25600]: 128: 269 -> 64, 512: 537 -> 208.
#include "prefill.hpp"

#include <algorithm>

namespace vt {
namespace {

typedef std::uint32_t u32x4 __attribute__((ext_vector_type(4)));

// One pair of the eight weights of a code word (columns c + 2p, c + 2p + 1, in
// column order). `word` holds biased nibbles u = q + 8; byte p is copied into
// both halves, a mask-and-or leaves 1024 + u0 in the low and 1024 + 16 u1 in
// the high half, one packed FMA makes both q exactly and one packed multiply
// rounds q * s once.
struct Q4Masks {
    std::uint32_t keep, one;
};
__device__ __forceinline__ Q4Masks q4_masks() {
    Q4Masks m{0x00F0000Fu, 0x64006400u};
    asm volatile("" : "+v"(m.keep), "+v"(m.one));  // kept in VGPRs: v_and_or_b32 takes no literal
    return m;
}
template <int P>
__device__ __forceinline__ half2v dequant_pair(std::uint32_t word, half2v s2, const Q4Masks& m) {
    constexpr std::uint32_t sel = 0x0C000C00u | P << 16 | P;
    const half2v scale = {static_cast<_Float16>(1.0f), static_cast<_Float16>(0.0625f)};
    const half2v bias = {static_cast<_Float16>(-1032.0f), static_cast<_Float16>(-72.0f)};
    const std::uint32_t bytes = __builtin_amdgcn_perm(word, word, sel);
    const half2v h = __builtin_bit_cast(half2v, (bytes & m.keep) | m.one);
    return __builtin_elementwise_fma(h, scale, bias) * s2;
}

__device__ __forceinline__ half8 join(const half2v (&p)[4]) {
    return half8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
}

// A wave's TI x TJ tiles of 16 tokens x 16 rows and the operands of one
// 32-column slice in registers.
template <int TI, int TJ>
struct Q4Tile {
    static constexpr int kTiles = TI * TJ, kPairs = 4 * TJ;
    static constexpr int kFirst = kTiles / 4;  // the next slice's words have arrived by then
    float4v y[TI][TJ];
    half8 fa[TI], fb[TJ];

    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j) y[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
    template <class Source>
    __device__ __forceinline__ void fill(const Source& src, const Q4Masks& masks) {
#pragma unroll
        for (int i = 0; i < TI; ++i) fa[i] = src.a(i);
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const std::uint32_t word = src.b(j);
            const half2v s2 = __builtin_bit_cast(half2v, src.scale(j));
            const half2v p[4] = {dequant_pair<0>(word, s2, masks), dequant_pair<1>(word, s2, masks),
                                 dequant_pair<2>(word, s2, masks), dequant_pair<3>(word, s2, masks)};
            fb[j] = join(p);
        }
    }
    // Multiplies the slice in registers; meanwhile the next slice's activation
    // fragments are read as their registers become free and its weights are
    // dequantized pair by pair. hook(t) runs before tile t.
    template <class Source, class Hook>
    __device__ __forceinline__ void slice(const Source& next, const Q4Masks& masks, Hook&& hook) {
        std::uint32_t word[TJ], scale[TJ];
        half2v p[TJ][4];
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            hook(t);
            const int i = t / TJ, j = t % TJ;
            y[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[i], fb[j], y[i][j], 0, 0, 0);
            if (j == TJ - 1) fa[i] = next.a(i);
            if (t < TJ) {
                word[t] = next.b(t);
                scale[t] = next.scale(t);
            }
            if (t >= kFirst) {
                constexpr int span = kTiles - kFirst;
                const int p0 = kPairs * (t - kFirst) / span, p1 = kPairs * (t - kFirst + 1) / span;
#pragma unroll
                for (int u = 0; u < kPairs; ++u) {
                    if (u < p0 || u >= p1) continue;
                    const half2v s2 = __builtin_bit_cast(half2v, scale[u / 4]);
                    p[u / 4][u % 4] = u % 4 == 0   ? dequant_pair<0>(word[u / 4], s2, masks)
                                      : u % 4 == 1 ? dequant_pair<1>(word[u / 4], s2, masks)
                                      : u % 4 == 2 ? dequant_pair<2>(word[u / 4], s2, masks)
                                                   : dequant_pair<3>(word[u / 4], s2, masks);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < TJ; ++j) fb[j] = join(p[j]);
    }
    // Partial sums of token tiles [I0, I0 + N) as fp32 rows of P floats.
    template <int I0, int N, int P>
    __device__ __forceinline__ void put(float* rows, int r, int q) const {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) rows[(i * 16 + 4 * q + e) * P + j * 16 + r] = y[I0 + i][j][e];
    }
};

// Where a wave's operands of one slice lie in LDS (byte addresses of its lane).
struct Q4Source {
    const unsigned char *pa, *pb, *ps;
    int a_stride, b_stride;  // bytes between tiles of 16 rows
    __device__ __forceinline__ half8 a(int i) const { return *reinterpret_cast<const half8*>(pa + i * a_stride); }
    __device__ __forceinline__ std::uint32_t b(int j) const {
        return *reinterpret_cast<const std::uint32_t*>(pb + j * b_stride);
    }
    __device__ __forceinline__ std::uint32_t scale(int j) const {
        return *reinterpret_cast<const std::uint32_t*>(ps + j * 64);
    }
};

template <int WT, int WN, int WK, int TI, int TJ>
struct Q4Geom {
    static_assert(WK == 2 || WK == 4, "a stage is one or two scale groups of 64 columns");
    static constexpr int kThreads = WT * WN * WK * 64;
    static constexpr int kTM = WT * TI * 16, kTN = WN * TJ * 16;
    static constexpr int kCols = 32 * WK;    // columns of a stage, one 32-column slice per K wave
    static constexpr int kAU = 4 * WK;       // 16-byte units of a staged activation row
    static constexpr int kBU = WK;           // 16-byte units of a staged row of codes
    static constexpr int kSG = WK / 2;       // scale groups of a stage
    static constexpr int kAPer = (kTM * kAU + kThreads - 1) / kThreads, kBPer = (kTN * kBU + kThreads - 1) / kThreads;
    static constexpr int kSPer = (kTN * kSG + kThreads - 1) / kThreads;
    // A buffer holds whole rounds of the threads' stores, so no store is guarded.
    static constexpr int kB = kAPer * kThreads * 16, kS = kB + kBPer * kThreads * 16;
    static constexpr int kStage = kS + kSPer * kThreads * 4;
    static constexpr int kPitch = kTN + 4;
    static constexpr int out_bytes(int oi) { return WK * WT * oi * 16 * kPitch * 4; }
    static constexpr int kOI = out_bytes(TI) <= 140 * 1024       ? TI
                               : TI % 2 == 0 && out_bytes(TI / 2) <= 140 * 1024 ? TI / 2
                               : TI % 4 == 0                                    ? TI / 4
                                                                                : 1;
    static constexpr int kLds = 2 * kStage > out_bytes(kOI) ? 2 * kStage : out_bytes(kOI);
    static_assert(TI % kOI == 0 && kLds <= 160 * 1024, "prefill tile exceeds LDS");
};

// Cooperative form: stages of 32 WK columns in two LDS buffers, one 32-column
// slice per K wave. While a stage is multiplied, the next one's operands are
// read, the one after is written to LDS and the one after that is requested.
template <int WT, int WN, int WK, int TI, int TJ>
__global__ __launch_bounds__(WT * WN * WK * 64, 2) void q4_prefill(const __half* __restrict__ x,
                                                                  const std::uint8_t* __restrict__ codes,
                                                                  const __half* __restrict__ scales,
                                                                  __half* __restrict__ out, int tokens, int n, int k,
                                                                  int padded, TileOrder order) {
    using G = Q4Geom<WT, WN, WK, TI, TJ>;
    constexpr int TM = G::kTM, TN = G::kTN, T = G::kThreads, AU = G::kAU, BU = G::kBU, SG = G::kSG;
    extern __shared__ uint4 q4p_lds[];
    auto* lds = reinterpret_cast<unsigned char*>(q4p_lds);
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wn = (wave / WK) % WN, wt = wave / (WK * WN);
    const int q = lane >> 4, r = lane & 15;
    const int tile = tile_of(order);
    if (tile < 0) return;
    const int t0 = tile % order.token_tiles * TM, n0 = tile / order.token_tiles * TN;

    const auto* a_base = reinterpret_cast<const char*>(x + static_cast<std::int64_t>(t0) * k);
    const auto* b_base = reinterpret_cast<const char*>(codes + static_cast<std::int64_t>(n0) * (padded / 2));
    const auto* s_base = reinterpret_cast<const char*>(scales + static_cast<std::int64_t>(n0) * (padded / 64));
    std::uint32_t a_off[G::kAPer], b_off[G::kBPer], s_off[G::kSPer];
    std::uint32_t a_put[G::kAPer], b_put[G::kBPer], s_put[G::kSPer];
#pragma unroll
    for (int u = 0; u < G::kAPer; ++u) {
        const int i = tid + u * T, row = i / AU;
        a_off[u] = 2u * (static_cast<std::uint32_t>(min(row, tokens - 1 - t0)) * k + 8 * (i % AU));
        a_put[u] = 16 * (row * AU + ((i % AU) ^ swizzle<AU>(row)));
    }
#pragma unroll
    for (int u = 0; u < G::kBPer; ++u) {
        const int i = tid + u * T, row = i / BU;
        b_off[u] = static_cast<std::uint32_t>(min(min(row, TN - 1), n - 1 - n0)) * (padded / 2) + 16 * (i % BU);
        b_put[u] = G::kB + 16 * (row * BU + ((i % BU) ^ swizzle<BU>(row)));
    }
#pragma unroll
    for (int u = 0; u < G::kSPer; ++u) {
        const int i = tid + u * T;
        s_off[u] = 2u * (static_cast<std::uint32_t>(min(min(i / SG, TN - 1), n - 1 - n0)) * (padded / 64) + i % SG);
        s_put[u] = G::kS + 4 * (i < TN * SG ? (i % SG) * TN + i / SG : i);
    }

    // The columns run in stages of KC. When K is not whole stages, the partial
    // one comes first (padded is whole stages, so only the activations are
    // masked): stage 0 then starts at column base `whole`, stage s > 0 at s - 1.
    constexpr int KC = G::kCols;
    const int whole = k / KC, edge = whole * KC < k ? 1 : 0, stages = whole + edge, last = max(whole - 1, 0);
    u32x4 st_a[G::kAPer], st_b[G::kBPer];
    unsigned short st_s[G::kSPer];
    auto load = [&](int stage) __attribute__((always_inline)) {
        const std::int64_t base = min(max(stage - edge, 0), last);
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u)
            st_a[u] = *reinterpret_cast<const u32x4*>(a_base + base * (2 * KC) + lane_offset(a_off[u]));
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u)
            st_b[u] = *reinterpret_cast<const u32x4*>(b_base + base * (KC / 2) + lane_offset(b_off[u]));
#pragma unroll
        for (int u = 0; u < G::kSPer; ++u)
            st_s[u] = *reinterpret_cast<const unsigned short*>(s_base + base * (2 * SG) + lane_offset(s_off[u]));
    };
    auto load_edge = [&]() __attribute__((always_inline)) {
        const std::int64_t base = whole;
        const int c0 = whole * KC;
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u) {
            const int col = 8 * ((tid + u * T) % AU);
            const u32x4 v = *reinterpret_cast<const u32x4*>(a_base + a_off[u] + 2 * static_cast<std::int64_t>(min(c0, k - 8 - col)));
            st_a[u] = c0 + col < k ? v : u32x4{0u, 0u, 0u, 0u};  // k % 8 == 0: a unit is all in or all out
        }
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u) st_b[u] = *reinterpret_cast<const u32x4*>(b_base + base * (KC / 2) + b_off[u]);
#pragma unroll
        for (int u = 0; u < G::kSPer; ++u)
            st_s[u] = *reinterpret_cast<const unsigned short*>(s_base + base * (2 * SG) + s_off[u]);
    };
    auto store = [&](int buf) __attribute__((always_inline)) {
        unsigned char* base = lds + buf * G::kStage;
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u) *reinterpret_cast<u32x4*>(base + a_put[u]) = st_a[u];
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u) *reinterpret_cast<u32x4*>(base + b_put[u]) = st_b[u] ^ 0x88888888u;  // q + 8
#pragma unroll
        for (int u = 0; u < G::kSPer; ++u)
            *reinterpret_cast<std::uint32_t*>(base + s_put[u]) = static_cast<std::uint32_t>(st_s[u]) * 0x10001u;
    };
    const std::uint32_t a_get = 16 * ((wt * TI * 16 + r) * AU + ((4 * wk + q) ^ swizzle<AU>(r)));
    const std::uint32_t b_get = G::kB + 16 * ((wn * TJ * 16 + r) * BU + (wk ^ swizzle<BU>(r))) + 4 * q;
    const std::uint32_t s_get = G::kS + 4 * ((wk / 2) * TN + wn * TJ * 16 + r);
    auto source = [&](int buf) __attribute__((always_inline)) {
        const unsigned char* base = lds + buf * G::kStage;
        return Q4Source{base + a_get, base + b_get, base + s_get, 256 * AU, 256 * BU};
    };

    const Q4Masks masks = q4_masks();
    Q4Tile<TI, TJ> m;
    m.clear();
    if (edge) {
        load_edge();
        store(0);
    } else {
        load(0);
        store(0);
    }
    if (stages > 1) {
        load(1);
        store(1);
    }
    if (whole == 0) {  // no whole stage: the loop's requests (never consumed) stay on column 0 of their rows
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u) a_off[u] -= 16 * ((tid + u * T) % AU);
    }
    load(2);
    __syncthreads();
    m.fill(source(0), masks);
    __syncthreads();
    constexpr int kStoreAt = TI * TJ / 8, kLoadAt = TI * TJ / 8 + 2;
    for (int sg = 0; sg < stages; ++sg) {
        m.slice(source((sg + 1) & 1), masks, [&](int t) __attribute__((always_inline)) {
            if (t == kStoreAt) store(sg & 1);
            if (t == kLoadAt) load(sg + 3);
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
struct Q4SplitGeom {
    static constexpr int kThreads = WK * 64;
    static constexpr int kTM = TI * 16, kTN = TJ * 16;
    static constexpr int kB = kTM * 128, kS = kB + kTN * 64, kWave = kS + 2 * 64 * 4;  // a 64-column step, codes of 128
    static constexpr int kPitch = kTN + 4;
    static constexpr int kOut = WK * kTM * kPitch * 4;
    static constexpr int kLds = WK * kWave > kOut ? WK * kWave : kOut;
    static_assert(kTN <= 64 && kLds <= 160 * 1024, "split tile exceeds LDS");
};

// Split form: every wave computes the whole tile over its own 128-column
// chunks through its own LDS region; no barrier before the final sum.
template <int WK, int TI, int TJ>
__global__ __launch_bounds__(WK * 64, 2) void q4_prefill_split(const __half* __restrict__ x,
                                                              const std::uint8_t* __restrict__ codes,
                                                              const __half* __restrict__ scales,
                                                              __half* __restrict__ out, int tokens, int n, int k,
                                                              int padded, TileOrder order) {
    using G = Q4SplitGeom<WK, TI, TJ>;
    constexpr int TM = G::kTM, TN = G::kTN, kA = 2 * TI, kB = TJ;
    extern __shared__ uint4 q4p_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, r = lane & 15;
    const int tile = tile_of(order);
    if (tile < 0) return;
    const int t0 = tile % order.token_tiles * TM, n0 = tile / order.token_tiles * TN;
    const int chunks = padded / 128;
    auto* lds = reinterpret_cast<unsigned char*>(q4p_lds) + wave * G::kWave;

    const Q4Masks masks = q4_masks();
    Q4Tile<TI, TJ> m;
    m.clear();
    if (wave < chunks) {
        const auto* a_base = reinterpret_cast<const char*>(x + static_cast<std::int64_t>(t0) * k);
        const auto* b_base = reinterpret_cast<const char*>(codes + static_cast<std::int64_t>(n0) * (padded / 2));
        const auto* s_base = reinterpret_cast<const char*>(scales + static_cast<std::int64_t>(n0) * (padded / 64));
        // Activation unit u of a lane: row lane / 8 + 8 u, unit lane % 8 of the step's 128 bytes; code unit u:
        // row lane / 4 + 16 u, unit lane % 4 of the chunk's 64 bytes; scales: row lane.
        std::uint32_t a_off[kA], b_off[kB], s_off;
#pragma unroll
        for (int u = 0; u < kA; ++u)
            a_off[u] = 2u * (static_cast<std::uint32_t>(min(lane / 8 + 8 * u, tokens - 1 - t0)) * k + 8 * (lane % 8));
#pragma unroll
        for (int u = 0; u < kB; ++u)
            b_off[u] = static_cast<std::uint32_t>(min(lane / 4 + 16 * u, n - 1 - n0)) * (padded / 2) + 16 * (lane % 4);
        s_off = 2u * static_cast<std::uint32_t>(min(lane, n - 1 - n0)) * (padded / 64);
        u32x4 st_a[kA], st_b[kB];
        std::uint32_t st_s;
        auto load_b = [&](std::int64_t c) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < kB; ++u) st_b[u] = *reinterpret_cast<const u32x4*>(b_base + c * 64 + lane_offset(b_off[u]));
            st_s = *reinterpret_cast<const std::uint32_t*>(s_base + c * 4 + lane_offset(s_off));
        };
        auto load_a = [&](std::int64_t c, int sub) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < kA; ++u)
                st_a[u] = *reinterpret_cast<const u32x4*>(a_base + c * 256 + sub * 128 + lane_offset(a_off[u]));
        };
        // The last chunk: columns past k are zero (k % 8 == 0: a unit is all in or all out).
        auto load_edge = [&](int c, int sub) __attribute__((always_inline)) {
            const int c0 = c * 128 + sub * 64, col = 8 * (lane % 8);
#pragma unroll
            for (int u = 0; u < kA; ++u) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(a_base + a_off[u] + 2 * static_cast<std::int64_t>(min(c0, k - 8 - col)));
                st_a[u] = c0 + col < k ? v : u32x4{0u, 0u, 0u, 0u};
            }
        };
        // Rows 8 apart alternate between two swizzles.
        std::uint32_t a_put[2];
#pragma unroll
        for (int odd = 0; odd < 2; ++odd) a_put[odd] = 16 * ((lane / 8) * 8 + ((lane % 8) ^ swizzle<8>(lane / 8 + 8 * odd)));
        const std::uint32_t b_put = G::kB + 16 * ((lane / 4) * 4 + ((lane % 4) ^ swizzle<4>(lane / 4)));
        auto store_a = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int u = 0; u < kA; ++u) *reinterpret_cast<u32x4*>(lds + a_put[u & 1] + u * 1024) = st_a[u];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        };
        auto store_b = [&]() __attribute__((always_inline)) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int u = 0; u < kB; ++u) *reinterpret_cast<u32x4*>(lds + b_put + u * 1024) = st_b[u] ^ 0x88888888u;  // q + 8
            *reinterpret_cast<std::uint32_t*>(lds + G::kS + 4 * lane) = (st_s & 0xffffu) * 0x10001u;
            *reinterpret_cast<std::uint32_t*>(lds + G::kS + 256 + 4 * lane) = (st_s >> 16) * 0x10001u;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        };
        std::uint32_t a_get[2], b_get[4];
#pragma unroll
        for (int g = 0; g < 2; ++g) a_get[g] = 16 * (r * 8 + ((4 * g + q) ^ swizzle<8>(r)));
#pragma unroll
        for (int g = 0; g < 4; ++g) b_get[g] = G::kB + 16 * (r * 4 + (g ^ swizzle<4>(r))) + 4 * q;
        auto source = [&](int g) __attribute__((always_inline)) {  // slice g of the chunk
            return Q4Source{lds + a_get[g & 1], lds + b_get[g], lds + G::kS + 256 * (g / 2) + 4 * r, 2048, 1024};
        };

        // The wave's chunks run from the last one down, so only the prologue
        // sees the edge; requests past the wave's last chunk go to chunk 0 and
        // are never consumed. The LDS region holds one step of activations and
        // one chunk of codes: a step is written over the previous one after
        // its last reads are issued (a wave's LDS accesses stay in order).
        int c = chunks - 1 - wave;
        load_b(c);
        store_b();
        if (c == chunks - 1) {
            load_edge(c, 0);
            store_a();
            load_edge(c, 1);
        } else {
            load_a(c, 0);
            store_a();
            load_a(c, 1);
        }
        load_b(max(c - WK, 0));
        m.fill(source(0), masks);
        for (; c >= 0; c -= WK) {
            const int next = max(c - WK, 0), after = max(c - 2 * WK, 0);
            each_slot<4>([&](auto g) __attribute__((always_inline)) {
                m.slice(source((g + 1) % 4), masks, [&](int t) __attribute__((always_inline)) {
                    if (g == 1 && t == 0) {
                        store_a();
                        load_a(next, 0);
                    }
                    if (g == 3 && t == 0) {
                        store_a();
                        store_b();
                        load_a(next, 1);
                        load_b(after);
                    }
                });
            });
        }
    }

    auto* o_lds = reinterpret_cast<float*>(q4p_lds);
    constexpr int P = G::kPitch;
    __syncthreads();
    m.template put<0, TI, P>(o_lds + wave * TM * P, r, q);
    __syncthreads();
    store_partials<WK, TM, TN, P, G::kThreads>(o_lds, out, tokens, n, n0, [&](int row) { return t0 + row; });
}

struct Q4Operands {
    const __half* x;
    const std::uint8_t* codes;
    const __half* scales;
    __half* out;
    int tokens, n, k, padded;
};

template <int WT, int WN, int WK, int TI, int TJ>
void launch_coop(const Q4Operands& o, hipStream_t stream) {
    using G = Q4Geom<WT, WN, WK, TI, TJ>;
    const auto kernel = q4_prefill<WT, WN, WK, TI, TJ>;
    const TileOrder order = tile_order(o.tokens, G::kTM, o.n, G::kTN);
    static LdsLimit limit;
    limit.raise(kernel, G::kLds);
    kernel<<<8 * order.per_xcd, G::kThreads, G::kLds, stream>>>(o.x, o.codes, o.scales, o.out, o.tokens, o.n, o.k,
                                                               o.padded, order);
}

template <int WK, int TI, int TJ>
void launch_split(const Q4Operands& o, hipStream_t stream) {
    using G = Q4SplitGeom<WK, TI, TJ>;
    const auto kernel = q4_prefill_split<WK, TI, TJ>;
    const TileOrder order = tile_order(o.tokens, G::kTM, o.n, G::kTN);
    static LdsLimit limit;
    limit.raise(kernel, G::kLds);
    kernel<<<8 * order.per_xcd, G::kThreads, G::kLds, stream>>>(o.x, o.codes, o.scales, o.out, o.tokens, o.n, o.k,
                                                               o.padded, order);
}

}  // namespace

// Runs the projection and returns 0, or launches nothing and returns the tile of
// row_prefill that is the fastest for this shape (4: 128 tokens x 128 rows; 5, 6
// and 7: 256 tokens x 32 times that many rows). Operands are admitted by the
// caller; rows of more than kNarrowK columns, past the 32-bit lane offsets, are
// left to row_prefill's own rule (-1).
int q4_prefill_launch(const __half* x, const std::uint8_t* codes, const __half* scales, __half* out, int tokens, int n,
                      int k, int padded, hipStream_t stream) {
    if (k > kNarrowK) return -1;
    const Q4Operands o{x, codes, scales, out, tokens, n, k, padded};
    // The tiling with the least predicted time; the last four are row_prefill's,
    // whose 256-token tiles read fewer LDS bytes per MFMA and win where whole
    // rounds of them fill the chip (2048 tokens x 34816 rows: 736 us against
    // 885), and whose 128 x 128 tile, two workgroups to a CU, wins where K is
    // short (128 tokens x 34816 rows x 1024: 26 us in the others, 21). The
    // constants are a fit to 770 shapes (33-8192 tokens, 256-151936 rows,
    // 64-25600 columns; each candidate timed on each shape on MI355X): the choice
    // is within 12% of the fastest candidate on every one of them and 0.3% on
    // average.
    constexpr PrefillTiling kTilings[12] = {
        {128, 128, 1, 0.0, 6.71, 7.70, 7.70},   {64, 128, 1, 0.8, 4.25, 6.10, 6.10},    {64, 64, 1, 1.4, 2.85, 3.36, 3.36},
        {64, 64, 2, 2.1, 3.01, 3.40, 6.13},     {48, 64, 2, 2.7, 1.38, 2.59, 5.08},     {48, 64, 1, 0.7, 3.53, 2.43, 2.43},
        {32, 64, 1, 3.0, 0.92, 2.20, 2.20},     {32, 32, 1, 1.3, 1.08, 1.76, 1.76},     {128, 128, 2, 1.3, 2.95, 9.09, 17.27},
        {256, 160, 1, 0.0, 7.58, 19.63, 19.63}, {256, 192, 1, 1.6, 8.60, 21.28, 21.28}, {256, 224, 1, 0.7, 7.86, 23.88, 23.88}};
    // (Past row_prefill's launch grid of 65535 token tiles, the forms here take every shape.)
    int best = tokens <= 65535 * 128 ? fastest_tiling(kTilings, tokens, n, k) : 0;
    if (best >= 2 && k < 128) best = 8;  // the split form needs one whole chunk
    if (best >= 8) return best - 4;
    switch (best) {
        case 0: launch_coop<1, 2, 4, 8, 4>(o, stream); break;
        case 1: launch_coop<1, 2, 4, 4, 4>(o, stream); break;
        case 2: launch_split<8, 4, 4>(o, stream); break;
        case 3: launch_split<4, 4, 4>(o, stream); break;
        case 4: launch_split<4, 3, 4>(o, stream); break;
        case 5: launch_split<8, 3, 4>(o, stream); break;
        case 6: launch_split<8, 2, 4>(o, stream); break;
        default: launch_split<8, 2, 2>(o, stream); break;
    }
    return 0;
}

}  // namespace vt
