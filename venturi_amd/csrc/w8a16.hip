// Q8 A16 projection for many tokens (prefill) on fp16 matrix cores: the
// "mfma" route above the decode kernels' 32 tokens.
//
// out[t][n] = fp16( sum_g D[t][n][g] * ws[n][g] ),  D = sum_{k in g} x[t][k] * code[n][k]
//
// Each 32-column group's D is one v_mfma_f32_16x16x32_f16 on the fp16
// activations and the int8 codes converted to fp16 exactly (every x * code
// product is exact in fp32); the group scale is one fp32 FMA per (t, n, g).
// A wave sums its groups in the order it visits them (cooperative: the partial
// stage first, then the others from column 0 up; split: its chunks from the
// last one down, a chunk's groups upwards), and the sums of the waves that
// split K are added in wave order. The order depends on shape and tiling only,
// so outputs are deterministic and agree with the canonical order
// (blocks.cu:306-321) to fp32 association, like the decode route.
//
// Two forms (prefill.hpp), chosen per shape by a measured time model:
// * cooperative (q8_prefill): WT x WN x WK waves compute (WT*TI*16) tokens x
//   (WN*TJ*16) rows; a stage is WK groups, staged in two LDS buffers
//   (activations as fp16, codes biased to unsigned), one group per K wave, one
//   barrier per stage. For grids that fill the chip; with short rows its
//   tilings of four waves that do not split K (64 x 128 and 128 x 128), which
//   need no sum and leave room for two to four workgroups per CU.
// * split (q8_prefill_split): each of WK waves computes the whole TI*16 x TJ*16
//   tile over its own 128-column chunks through its own LDS region; no barrier
//   before the sum. For the small grids of short prompts, where it fills the
//   CUs with K instead of tiles.
//
// What binds them: no unit alone. Per 16 x 16 tile and group there are one MFMA
// and four scaling FMAs, plus a tile row's share of the code conversion, so
// both forms issue a tile's MFMA four tiles before its FMAs, replace each
// activation fragment by the next group's as soon as its last MFMA is issued,
// and pin that order with scheduling barriers. Counters, [34816 x 5120] at 2048
// tokens / [7168 x 5120] at 200: matrix cores busy 33 / 19% of the time, VALU
// at most 56 / 38% (4 cycles per instruction; an FMA measured 2.7 in a dense
// loop), LDS active 31 / 30%, waves waiting 35 / 32% of theirs. The shares add
// up to about the whole: with the two waves per SIMD that the registers leave
// room for, matrix, VALU and LDS work still run largely one after another.
// Measured on MI355X against one workgroup of 8 waves with a barrier per group
// (the form this replaces), us:
//   tokens x [7168 x 5120]:  64: 74.6 -> 17.0, 200: 76.5 -> 33.3, 512: 77.3 -> 55,
//     1024: 137 -> 101; [5120 x 17408]: 64: 255 -> 43, 512: 267 -> 178;
//   [34816 x 5120], 2048 tokens: 1210 -> 1030 (710 TFLOP/s).
// Up to about 256 columns over 16384 or more rows, and at 100-128 tokens over
// 34816 rows of 64-512, it is up to 1.14 (at 64 columns 1.24) times the time of
// the replaced form: prologue and output, not the K loop, are the time there.
#include "prefill.hpp"

#include <algorithm>

namespace vt {
namespace {

// Eight biased codes u = c + 128 (one MFMA B fragment of a lane) -> fp16 c.
__device__ __forceinline__ half8 codes8_to_fp16(const uint2 w) {
    const half2v bias = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
    const std::uint32_t words[2] = {w.x, w.y};
    half8 h;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const half2v a = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, words[i], 0x05010400u)) + bias;
        const half2v b = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, words[i], 0x05030402u)) + bias;
        h[4 * i] = a[0]; h[4 * i + 1] = a[1]; h[4 * i + 2] = b[0]; h[4 * i + 3] = b[1];
    }
    return h;
}

template <int WT, int WN, int WK, int TI, int TJ>
struct PrefillGeom {
    static constexpr int kThreads = WT * WN * WK * 64;
    static constexpr int kTM = WT * TI * 16;   // tokens per workgroup
    static constexpr int kTN = WN * TJ * 16;   // weight rows per workgroup
    static constexpr int kGroups = WK;         // groups of 32 columns per stage, one per wave of a K set
    static constexpr int kAU = 4 * kGroups;    // 16-byte units of a staged activation row (fp16)
    static constexpr int kBU = 2 * kGroups;    // 16-byte units of a staged weight row (int8 codes)
    static constexpr int kAUnits = kTM * kAU;
    static constexpr int kBUnits = kTN * kBU;
    static constexpr int kSUnits = kTN * kGroups;  // scales of a stage
    static constexpr int kAPer = (kAUnits + kThreads - 1) / kThreads;
    static constexpr int kBPer = (kBUnits + kThreads - 1) / kThreads;
    static constexpr int kSPer = (kSUnits + kThreads - 1) / kThreads;
    // A buffer holds whole rounds of the threads' stores, so no store is guarded.
    static constexpr int kABytes = kAPer * kThreads * 16, kBBytes = kBPer * kThreads * 16, kSBytes = kSPer * kThreads * 4;
    static constexpr int kStageBytes = kABytes + kBBytes + kSBytes;
    // Output: the WK partial sums of OI token tiles of every wave at a time, fp32 rows of kTN + 4. Where one wave runs
    // the whole K, up to 36 KB of them at once: four workgroups still share a CU.
    static constexpr int kPitch = kTN + 4;
    static constexpr int out_bytes(int oi) { return WK * WT * oi * 16 * kPitch * 4; }
    static constexpr int kOI = out_bytes(TI) <= 2 * kStageBytes || (WK == 1 && out_bytes(TI) <= 36 * 1024) ? TI
                               : TI % 2 == 0 && out_bytes(TI / 2) <= 2 * kStageBytes ? TI / 2
                               : TI % 4 == 0 && out_bytes(TI / 4) <= 2 * kStageBytes ? TI / 4
                                                                                      : 1;
    static constexpr int kLds = 2 * kStageBytes > out_bytes(kOI) ? 2 * kStageBytes : out_bytes(kOI);
    static_assert(TI % kOI == 0 && kLds <= 160 * 1024, "prefill tile exceeds LDS");
};

// PF stages are in flight in registers; Off is the type of the lane offsets
// (32 bits up to kNarrowK columns).
template <int WT, int WN, int WK, int TI, int TJ, int PF, class Off>
__global__ __launch_bounds__(WT * WN * WK * 64, 2) void q8_prefill(const __half* __restrict__ x,
                                                                  const std::int8_t* __restrict__ codes,
                                                                  const __half* __restrict__ scales,
                                                                  __half* __restrict__ out, int tokens, int n, int k,
                                                                  int padded, int groups, TileOrder order) {
    using G = PrefillGeom<WT, WN, WK, TI, TJ>;
    constexpr int TM = G::kTM, TN = G::kTN, T = G::kThreads, AU = G::kAU, BU = G::kBU, KG = G::kGroups;
    extern __shared__ uint4 q8p_lds[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wk = wave % WK, wn = (wave / WK) % WN, wt = wave / (WK * WN);
    const int q = lane >> 4, r = lane & 15;
    const int tile = tile_of(order);
    if (tile < 0) return;
    const int t0 = tile % order.token_tiles * TM, n0 = tile / order.token_tiles * TN;
    const int stages = (groups + KG - 1) / KG;
    auto* lds = reinterpret_cast<unsigned char*>(q8p_lds);
    Off a_off[G::kAPer], b_off[G::kBPer], s_off[G::kSPer];
    const auto* a_base = reinterpret_cast<const char*>(x + static_cast<std::int64_t>(t0) * k);
    const auto* b_base = reinterpret_cast<const char*>(codes + static_cast<std::int64_t>(n0) * padded);
    const auto* s_base = reinterpret_cast<const char*>(scales + static_cast<std::int64_t>(n0) * (padded / 32));
#pragma unroll
    for (int u = 0; u < G::kAPer; ++u) {
        const int i = tid + u * T;
        a_off[u] = 2u * (static_cast<Off>(min(i / AU, tokens - 1 - t0)) * k + 8 * (i % AU));
    }
#pragma unroll
    for (int u = 0; u < G::kBPer; ++u) {
        const int i = tid + u * T;
        b_off[u] = static_cast<Off>(min(i / BU, n - 1 - n0)) * padded + 16 * (i % BU);
    }
#pragma unroll
    for (int u = 0; u < G::kSPer; ++u) {
        const int i = tid + u * T;
        s_off[u] = 2u * (static_cast<Off>(min(i / KG, n - 1 - n0)) * (padded / 32) + i % KG);
    }
    // The columns run in stages of 32 KG. When K is not whole stages, the
    // partial one comes first, so that only the prologue masks and clamps:
    // stage 0 then starts at the last column base, stage s > 0 at s - 1.
    constexpr int KC = 32 * KG;
    const int whole = k / KC, first = whole < stages ? whole : 0, shift = whole < stages ? 1 : 0;
    constexpr int kSlots = PF < 2 ? 2 : PF;  // PF stages in flight, two in the prologue
    uint4 st_a[kSlots][G::kAPer], st_b[kSlots][G::kBPer];
    unsigned short st_s[kSlots][G::kSPer];
    // Loads stage columns [c0, c0 + KC), all of them real ones.
    auto load = [&](int base, auto slot) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u)
            st_a[slot][u] = *reinterpret_cast<const uint4*>(a_base + static_cast<std::int64_t>(base) * (2 * KC) + lane_offset(a_off[u]));
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u)
            st_b[slot][u] = *reinterpret_cast<const uint4*>(b_base + static_cast<std::int64_t>(base) * KC + lane_offset(b_off[u]));
#pragma unroll
        for (int u = 0; u < G::kSPer; ++u)
            st_s[slot][u] = *reinterpret_cast<const unsigned short*>(s_base + static_cast<std::int64_t>(base) * (2 * KG) +
                                                               lane_offset(s_off[u]));
    };
    auto load_edge = [&](int base, auto slot) __attribute__((always_inline)) {
        const int c0 = base * KC;
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u) {
            const int col = 8 * ((tid + u * T) % AU);
            const uint4 v = *reinterpret_cast<const uint4*>(a_base + a_off[u] + 2 * static_cast<std::int64_t>(min(c0, k - 8 - col)));
            st_a[slot][u] = c0 + col < k ? v : make_uint4(0u, 0u, 0u, 0u);  // k % 8 == 0: a unit is all in or all out
        }
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u) {
            const int col = 16 * ((tid + u * T) % BU);
            st_b[slot][u] = *reinterpret_cast<const uint4*>(b_base + b_off[u] + static_cast<std::int64_t>(min(c0, padded - 16 - col)));
        }
#pragma unroll
        for (int u = 0; u < G::kSPer; ++u) {
            const int g = (tid + u * T) % KG;
            const unsigned short v = *reinterpret_cast<const unsigned short*>(s_base + s_off[u] + 2 * static_cast<std::int64_t>(min(base * KG, groups - 1 - g)));
            st_s[slot][u] = base * KG + g < groups ? v : 0;  // groups past the last one carry scale 0
        }
    };
    // LDS offsets: a store unit's, and those of the lane's fragments (rows 16
    // apart share a swizzle, so tiles are whole strides apart).
    std::uint32_t a_put[G::kAPer], b_put[G::kBPer], s_put[G::kSPer];
#pragma unroll
    for (int u = 0; u < G::kAPer; ++u) {
        const int i = tid + u * T, row = i / AU;
        a_put[u] = 16 * (row * AU + ((i % AU) ^ swizzle<AU>(row)));
    }
#pragma unroll
    for (int u = 0; u < G::kBPer; ++u) {
        const int i = tid + u * T, row = i / BU;
        b_put[u] = G::kABytes + 16 * (row * BU + ((i % BU) ^ swizzle<BU>(row)));
    }
#pragma unroll
    for (int u = 0; u < G::kSPer; ++u) {
        const int i = tid + u * T;
        s_put[u] = G::kABytes + G::kBBytes + 4 * (i < G::kSUnits ? (i % KG) * TN + i / KG : i);
    }
    const std::uint32_t a_get = 16 * ((wt * TI * 16 + r) * AU + ((4 * wk + q) ^ swizzle<AU>(r)));
    const std::uint32_t b_get =
        G::kABytes + 16 * ((wn * TJ * 16 + r) * BU + ((2 * wk + (q >> 1)) ^ swizzle<BU>(r))) + 8 * (q & 1);
    const std::uint32_t s_get = G::kABytes + G::kBBytes + 4 * (wk * TN + wn * TJ * 16 + r);
    auto store = [&](int buf, auto slot) __attribute__((always_inline)) {
        unsigned char* base = lds + buf * G::kStageBytes;
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u) *reinterpret_cast<uint4*>(base + a_put[u]) = st_a[slot][u];
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u) {
            const uint4 v = st_b[slot][u];  // biased: code + 128
            *reinterpret_cast<uint4*>(base + b_put[u]) =
                make_uint4(v.x ^ 0x80808080u, v.y ^ 0x80808080u, v.z ^ 0x80808080u, v.w ^ 0x80808080u);
        }
#pragma unroll
        for (int u = 0; u < G::kSPer; ++u)
            *reinterpret_cast<float*>(base + s_put[u]) = __half2float(__ushort_as_half(st_s[slot][u]));
    };
    half8 fa[TI];
    uint2 rb[TJ];
    float ws[TJ];
    auto read_a = [&](int buf, int i) __attribute__((always_inline)) {
        fa[i] = *reinterpret_cast<const half8*>(lds + buf * G::kStageBytes + a_get + i * 256 * AU);
    };
    auto read_b = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            rb[j] = *reinterpret_cast<const uint2*>(lds + buf * G::kStageBytes + b_get + j * 256 * BU);
            ws[j] = *reinterpret_cast<const float*>(lds + buf * G::kStageBytes + s_get + j * 64);
        }
    };

    float4v y[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) y[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    // Stage s is multiplied from registers while stage s + 1 is read from LDS
    // (each activation fragment as soon as its register is free), stage s + 2
    // is written to LDS and stage s + 3 is requested from memory.
    const int last = max(whole - 1, 0);  // the last whole stage's column base
    // The first two stages are requested together: for short rows the prologue
    // is most of the time.
    load_edge(first, Slot<0>{});
    if (whole == 0) {
        // The partial stage is the only one: the other requests (never
        // consumed) stay on column 0 of their rows.
#pragma unroll
        for (int u = 0; u < G::kAPer; ++u) a_off[u] -= 16u * ((tid + u * T) % AU);
#pragma unroll
        for (int u = 0; u < G::kBPer; ++u) b_off[u] -= 16u * ((tid + u * T) % BU);
#pragma unroll
        for (int u = 0; u < G::kSPer; ++u) s_off[u] -= 2u * ((tid + u * T) % KG);
    }
    load(min(1 - shift, last), Slot<1>{});
    store(0, Slot<0>{});
    store(1, Slot<1>{});
    each_slot<PF>([&](auto p) __attribute__((always_inline)) { load(min(2 + p - shift, last), p); });
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TI; ++i) read_a(0, i);
    read_b(0);
    __syncthreads();
    constexpr int kTiles = TI * TJ, kAhead = kTiles < 4 ? 1 : 4;
    constexpr int kStoreAt = kTiles / 4, kLoadAt = kTiles / 4 + 2, kReadB = TJ + kTiles / 4;
    auto step = [&](int sg, auto slot) __attribute__((always_inline)) {
        const int next = (sg + 1) & 1;
        const float4v zero = {0.0f, 0.0f, 0.0f, 0.0f};
        half8 fb[TJ];
        float wj[TJ];
#pragma unroll
        for (int j = 0; j < TJ; ++j) wj[j] = ws[j];
        // Tile t's MFMA is issued kAhead tiles before its four scaling FMAs, so
        // the matrix cores run under the wave's own VALU work.
        float4v d[kAhead];
#pragma unroll
        for (int t = 0; t < kTiles + kAhead; ++t) {
            if (t >= kAhead) {
                const int f = t - kAhead, i = f / TJ, j = f % TJ;
#pragma unroll
                for (int e = 0; e < 4; ++e) y[i][j][e] = fmaf(d[f % kAhead][e], wj[j], y[i][j][e]);
            }
            if (t < TJ) fb[t] = codes8_to_fp16(rb[t]);
            if (t < kTiles) {
                d[t % kAhead] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[t / TJ], fb[t % TJ], zero, 0, 0, 0);
                if (t % TJ == TJ - 1) read_a(next, t / TJ);
            }
            if (t == kStoreAt) store(sg & 1, slot);
            if (t == kLoadAt) load(min(sg + 2 + PF - shift, last), slot);
            if (t == kReadB) read_b(next);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    };
    int sg = 0;
    for (; sg + PF <= stages; sg += PF) {
        each_slot<PF>([&](auto p) __attribute__((always_inline)) { step(sg + p, p); });
    }
    each_slot<PF - 1>([&](auto p) __attribute__((always_inline)) {
        if (sg + p < stages) step(sg + p, p);
    });

    // The partial sums of the WK waves through LDS, OI token tiles of every
    // wave at a time.
    auto* o_lds = reinterpret_cast<float*>(q8p_lds);
    constexpr int OI = G::kOI, P = G::kPitch, kRows = WT * OI * 16;
#pragma unroll
    for (int c = 0; c < TI / OI; ++c) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < OI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o_lds[(wk * kRows + (wt * OI + i) * 16 + 4 * q + e) * P + wn * TJ * 16 + j * 16 + r] = y[c * OI + i][j][e];
        __syncthreads();
        store_partials<WK, kRows, TN, P, T>(o_lds, out, tokens, n, n0, [&](int row) {
            return t0 + (row / (OI * 16)) * TI * 16 + c * OI * 16 + row % (OI * 16);
        });
    }
}

template <int WT, int WN, int WK, int TI, int TJ, int PF, class Off = std::uint32_t>
void launch_prefill(const __half* x, const std::int8_t* codes, const __half* scales, __half* out, int tokens, int n,
                    int k, int padded, hipStream_t stream) {
    using G = PrefillGeom<WT, WN, WK, TI, TJ>;
    const auto kernel = q8_prefill<WT, WN, WK, TI, TJ, PF, Off>;
    const TileOrder order = tile_order(tokens, G::kTM, n, G::kTN);
    static LdsLimit limit;
    limit.raise(kernel, G::kLds);
    kernel<<<8 * order.per_xcd, G::kThreads, G::kLds, stream>>>(x, codes, scales, out, tokens, n, k, padded,
                                                               (k + 31) / 32, order);
}

template <int WK, int TI, int TJ>
struct SplitGeom {
    static constexpr int kThreads = WK * 64;
    static constexpr int kTM = TI * 16, kTN = TJ * 16;
    static constexpr int kA = 2 * TI;                   // 16-byte activation loads of a lane per step (64 columns)
    static constexpr int kB = TJ;                       // 16-byte code loads of a lane per step
    static constexpr int kABytes = kTM * 128, kBBytes = kTN * 64, kSBytes = 4 * 64 * 4;
    static constexpr int kWave = kABytes + kBBytes + kSBytes;
    static constexpr int kPitch = kTN + 4;
    static constexpr int kOut = WK * kTM * kPitch * 4;
    static constexpr int kLds = WK * kWave > kOut ? WK * kWave : kOut;
    static_assert(kTN <= 64 && kLds <= 160 * 1024, "split tile exceeds LDS");
};

template <int WK, int TI, int TJ>
__global__ __launch_bounds__(WK * 64, 2) void q8_prefill_split(const __half* __restrict__ x,
                                                              const std::int8_t* __restrict__ codes,
                                                              const __half* __restrict__ scales,
                                                              __half* __restrict__ out, int tokens, int n, int k,
                                                              int padded, int groups, TileOrder order) {
    using G = SplitGeom<WK, TI, TJ>;
    constexpr int TM = G::kTM, TN = G::kTN;
    extern __shared__ uint4 q8p_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, r = lane & 15;
    const int tile = tile_of(order);
    if (tile < 0) return;
    const int t0 = tile % order.token_tiles * TM, n0 = tile / order.token_tiles * TN;
    const int chunks = padded / 128;
    auto* lds = reinterpret_cast<unsigned char*>(q8p_lds) + wave * G::kWave;

    float4v y[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) y[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

    if (wave < chunks) {
        // Lane offsets of the loads: activation unit u is row lane / 8 + 8 u of
        // the tile, 16-byte unit lane % 8 of its 128 bytes; code unit u row
        // lane / 4 + 16 u, unit lane % 4 of its 64 bytes; scales row lane.
        std::uint32_t a_off[G::kA], b_off[G::kB], s_off;
        const auto* a_base = reinterpret_cast<const char*>(x + static_cast<std::int64_t>(t0) * k);
        const auto* b_base = reinterpret_cast<const char*>(codes + static_cast<std::int64_t>(n0) * padded);
        const auto* s_base = reinterpret_cast<const char*>(scales + static_cast<std::int64_t>(n0) * (padded / 32));
#pragma unroll
        for (int u = 0; u < G::kA; ++u)
            a_off[u] = 2u * (static_cast<std::uint32_t>(min(lane / 8 + 8 * u, tokens - 1 - t0)) * k + 8 * (lane % 8));
#pragma unroll
        for (int u = 0; u < G::kB; ++u)
            b_off[u] = static_cast<std::uint32_t>(min(lane / 4 + 16 * u, n - 1 - n0)) * padded + 16 * (lane % 4);
        s_off = 2u * static_cast<std::uint32_t>(min(lane, n - 1 - n0)) * (padded / 32);
        uint4 st_a[G::kA], st_b[G::kB];
        uint2 st_s;
        // Step `sub` (64 columns) of chunk c, all of them real columns.
        auto load = [&](int c, auto sub) __attribute__((always_inline)) {
            const std::int64_t c0 = static_cast<std::int64_t>(c) * 128 + sub * 64;
#pragma unroll
            for (int u = 0; u < G::kA; ++u) st_a[u] = *reinterpret_cast<const uint4*>(a_base + 2 * c0 + lane_offset(a_off[u]));
#pragma unroll
            for (int u = 0; u < G::kB; ++u) st_b[u] = *reinterpret_cast<const uint4*>(b_base + c0 + lane_offset(b_off[u]));
            if constexpr (sub == 0)
                st_s = *reinterpret_cast<const uint2*>(s_base + 8 * static_cast<std::int64_t>(c) + lane_offset(s_off));
        };
        // The same for the last chunk: columns past k are zero (k % 8 == 0: a
        // unit is all in or all out), groups past the last one carry scale 0.
        auto load_edge = [&](int c, auto sub) __attribute__((always_inline)) {
            load(0, sub);
            const int c0 = c * 128 + sub * 64, col = c0 + 8 * (lane % 8);
#pragma unroll
            for (int u = 0; u < G::kA; ++u) {
                const uint4 v = *reinterpret_cast<const uint4*>(
                    a_base + a_off[u] + 2 * static_cast<std::int64_t>(min(c0, k - 8 - 8 * (lane % 8))));
                st_a[u] = col < k ? v : make_uint4(0u, 0u, 0u, 0u);
            }
#pragma unroll
            for (int u = 0; u < G::kB; ++u) st_b[u] = *reinterpret_cast<const uint4*>(b_base + c0 + b_off[u]);
            if constexpr (sub == 0) {
                const uint2 v = *reinterpret_cast<const uint2*>(s_base + 8 * static_cast<std::int64_t>(c) + s_off);
                const int real = groups - 4 * c;  // 1 .. 4
                st_s.x = real >= 2 ? v.x : v.x & 0xffffu;
                st_s.y = real >= 4 ? v.y : real == 3 ? v.y & 0xffffu : 0u;
            }
        };
        const std::uint32_t a_put = 16 * ((lane / 8) * 8 + ((lane % 8) ^ swizzle<8>(lane / 8)));
        const std::uint32_t a_put_odd = 16 * ((lane / 8) * 8 + ((lane % 8) ^ swizzle<8>(lane / 8 + 8)));
        const std::uint32_t b_put = G::kABytes + 16 * ((lane / 4) * 4 + ((lane % 4) ^ swizzle<4>(lane / 4)));
        const std::uint32_t s_put = G::kABytes + G::kBBytes + 4 * lane;
        std::uint32_t a_get[2], b_get[2];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            a_get[g] = 16 * (r * 8 + ((4 * g + q) ^ swizzle<8>(r)));
            b_get[g] = G::kABytes + 16 * (r * 4 + ((2 * g + (q >> 1)) ^ swizzle<4>(r))) + 8 * (q & 1);
        }
        const std::uint32_t s_get = G::kABytes + G::kBBytes + 4 * r;
        auto store = [&](auto sub) __attribute__((always_inline)) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int u = 0; u < G::kA; ++u)
                *reinterpret_cast<uint4*>(lds + (u & 1 ? a_put_odd : a_put) + u * 1024) = st_a[u];
#pragma unroll
            for (int u = 0; u < G::kB; ++u) {
                const uint4 v = st_b[u];  // biased: code + 128
                *reinterpret_cast<uint4*>(lds + b_put + u * 1024) =
                    make_uint4(v.x ^ 0x80808080u, v.y ^ 0x80808080u, v.z ^ 0x80808080u, v.w ^ 0x80808080u);
            }
            if constexpr (sub == 0) {
                const float f[4] = {half_lo(st_s.x), half_hi(st_s.x), half_lo(st_s.y), half_hi(st_s.y)};
#pragma unroll
                for (int g = 0; g < 4; ++g) *reinterpret_cast<float*>(lds + s_put + 256 * g) = f[g];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        };
        half8 fa[TI];
        uint2 rb[TJ];
        float ws[TJ];
        auto read_a = [&](int g, int i) __attribute__((always_inline)) {
            fa[i] = *reinterpret_cast<const half8*>(lds + a_get[g & 1] + i * 2048);
        };
        auto read_b = [&](int g) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                rb[j] = *reinterpret_cast<const uint2*>(lds + b_get[g & 1] + j * 1024);
                ws[j] = *reinterpret_cast<const float*>(lds + s_get + 256 * g + j * 64);
            }
        };

        // The wave's chunks run from the last one down, so only the prologue
        // sees the edge; requests past the wave's last chunk go to chunk 0 and
        // are never consumed.
        int c = chunks - 1 - wave;
        if (c == chunks - 1) {
            load_edge(c, Slot<0>{});
            store(Slot<0>{});
            load_edge(c, Slot<1>{});
        } else {
            load(c, Slot<0>{});
            store(Slot<0>{});
            load(c, Slot<1>{});
        }
#pragma unroll
        for (int i = 0; i < TI; ++i) read_a(0, i);
        read_b(0);
        constexpr int kTiles = TI * TJ, kAhead = kTiles < 5 ? 2 : 4;
        for (; c >= 0; c -= WK) {
            const int next = max(c - WK, 0);
            each_slot<4>([&](auto g) __attribute__((always_inline)) {
                // Group g of the chunk is multiplied from registers; each
                // activation fragment is replaced by the next group's as soon
                // as it is free. The LDS holds one step (two groups): after the
                // last reads of a step the next one is written over it (a
                // wave's LDS accesses stay in order, and no other wave sees
                // its region), and the one after that is requested.
                const float4v zero = {0.0f, 0.0f, 0.0f, 0.0f};
                half8 fb[TJ];
                float wj[TJ];
#pragma unroll
                for (int j = 0; j < TJ; ++j) wj[j] = ws[j];
                float4v d[kAhead];
#pragma unroll
                for (int t = 0; t < kTiles + kAhead; ++t) {
                    if (t >= kAhead) {
                        const int f = t - kAhead, i = f / TJ, j = f % TJ;
#pragma unroll
                        for (int e = 0; e < 4; ++e) y[i][j][e] = fmaf(d[f % kAhead][e], wj[j], y[i][j][e]);
                    }
                    if (t < TJ) fb[t] = codes8_to_fp16(rb[t]);
                    if (t == 0 && g == 1) {
                        store(Slot<1>{});
                        load(next, Slot<0>{});
                    }
                    if (t == 0 && g == 3) {
                        store(Slot<0>{});
                        load(next, Slot<1>{});
                    }
                    if (t < kTiles) {
                        d[t % kAhead] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[t / TJ], fb[t % TJ], zero, 0, 0, 0);
                        if (t % TJ == TJ - 1) read_a(g + 1, t / TJ);
                    }
                    if (t == TJ) read_b((g + 1) & 3);
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
        }
    }

    // The partial sums of the waves through LDS.
    auto* o_lds = reinterpret_cast<float*>(q8p_lds);
    constexpr int P = G::kPitch;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) o_lds[(wave * TM + i * 16 + 4 * q + e) * P + j * 16 + r] = y[i][j][e];
    __syncthreads();
    store_partials<WK, TM, TN, P, G::kThreads>(o_lds, out, tokens, n, n0, [&](int row) { return t0 + row; });
}

template <int WK, int TI, int TJ>
void launch_split(const __half* x, const std::int8_t* codes, const __half* scales, __half* out, int tokens, int n,
                  int k, int padded, hipStream_t stream) {
    using G = SplitGeom<WK, TI, TJ>;
    const auto kernel = q8_prefill_split<WK, TI, TJ>;
    const TileOrder order = tile_order(tokens, G::kTM, n, G::kTN);
    static LdsLimit limit;
    limit.raise(kernel, G::kLds);
    kernel<<<8 * order.per_xcd, G::kThreads, G::kLds, stream>>>(x, codes, scales, out, tokens, n, k, padded,
                                                               (k + 31) / 32, order);
}

// The exact two-term fp16 form of Q8 weights, for the dense route: row j of
// the shadow holds hi = fp16(q*s) in columns [0, k) and lo = q*s - hi in
// [k, 2k). q*s is exact in fp32 (an 8-bit integer times an 11-bit
// significand), hi is its RNE fp16 rounding, and the difference is a multiple
// of the scale's ulp smaller than half an ulp of hi, at most 8 significant
// bits, which fp16 (with its subnormals) holds exactly; so hi + lo == q*s for
// every scale below 516. At 516 and above 127*s rounds past 65504: hi becomes
// inf and lo -inf, and every output that row touches is NaN, never a finite
// wrong value. Thread: 8 columns of one row (k % 8 == 0).
__global__ __launch_bounds__(256) void q8_split(const std::int8_t* __restrict__ codes, const __half* __restrict__ scales,
                                                __half* __restrict__ shadow, int row0, int k, int padded) {
    const int c = (blockIdx.x * 256 + threadIdx.x) * 8;
    if (c >= k) return;
    const std::int64_t row = row0 + static_cast<std::int64_t>(blockIdx.y);
    const uint2 w = *reinterpret_cast<const uint2*>(codes + row * padded + c);
    const float s = __half2float(scales[row * (padded / 32) + c / 32]);
    const std::uint32_t words[2] = {w.x, w.y};
    std::uint32_t hi[4], lo[4];
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        float v[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
            v[j] = static_cast<float>(static_cast<std::int8_t>(words[(i + j) / 4] >> (8 * ((i + j) % 4)))) * s;
        const __half h0 = __float2half_rn(v[0]), h1 = __float2half_rn(v[1]);
        const __half l0 = __float2half_rn(v[0] - __half2float(h0)), l1 = __float2half_rn(v[1] - __half2float(h1));
        hi[i / 2] = static_cast<std::uint32_t>(__half_as_ushort(h0)) | static_cast<std::uint32_t>(__half_as_ushort(h1)) << 16;
        lo[i / 2] = static_cast<std::uint32_t>(__half_as_ushort(l0)) | static_cast<std::uint32_t>(__half_as_ushort(l1)) << 16;
    }
    __half* dst = shadow + static_cast<std::int64_t>(blockIdx.y) * 2 * k + c;
    *reinterpret_cast<uint4*>(dst) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    *reinterpret_cast<uint4*>(dst + k) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
}

// x [tokens][k] -> x2 [tokens][2k] = [x | x] (the activations of the dense
// route's doubled K). Thread: 8 halves (k % 8 == 0).
__global__ __launch_bounds__(256) void q8_dup_rows(const __half* __restrict__ x, __half* __restrict__ x2, int k) {
    const int c = (blockIdx.x * 256 + threadIdx.x) * 8;
    if (c >= k) return;
    const std::int64_t t = blockIdx.y;
    const uint4 v = *reinterpret_cast<const uint4*>(x + t * k + c);
    *reinterpret_cast<uint4*>(x2 + t * 2 * k + c) = v;
    *reinterpret_cast<uint4*>(x2 + t * 2 * k + k + c) = v;
}

}  // namespace

void q8_split_launch(const std::int8_t* codes, const __half* scales, void* shadow, int row0, int rows, int k,
                     int padded, hipStream_t stream) {
    require(k % 8 == 0 && rows > 0 && rows <= 65535 && padded == padded_k(k), "invalid Q8 split geometry");
    require(aligned(codes, 8) && aligned(scales, 2) && aligned(shadow, 16), "misaligned Q8 split operand");
    q8_split<<<dim3((k / 8 + 255) / 256, rows), 256, 0, stream>>>(codes, scales, static_cast<__half*>(shadow), row0, k,
                                                                 padded);
}

void q8_dup_launch(const void* x, void* x2, int tokens, int k, hipStream_t stream) {
    require(k % 8 == 0 && tokens > 0 && tokens <= 65535, "invalid activation geometry for the dense Q8 route");
    q8_dup_rows<<<dim3((k / 8 + 255) / 256, tokens), 256, 0, stream>>>(static_cast<const __half*>(x),
                                                                       static_cast<__half*>(x2), k);
}

void q8_prefill_launch(const void* x, const std::int8_t* codes, const __half* scales, void* out, int tokens, int n,
                       int k, int padded, int dtype, hipStream_t stream) {
    require(x && codes && scales && out, "null Q8 operand");
    require(tokens > 0 && n > 0 && k > 0 && padded == padded_k(k), "invalid Q8 geometry");
    require(static_cast<std::int64_t>(tokens) * n < INT32_MAX, "Q8 output count exceeds int32");
    require(dtype == kF16, "the Q8 prefill GEMM takes FP16 activations");
    require(k % 8 == 0 && aligned(x, 16), "the Q8 prefill GEMM needs k % 8 == 0 and 16-byte aligned x");
    require(aligned(codes, 16) && aligned(scales, 2) && aligned(out, 2), "misaligned Q8 operand");
    const auto* xp = static_cast<const __half*>(x);
    auto* op = static_cast<__half*>(out);
    if (k > kNarrowK) {  // rows too long for 32-bit lane offsets
        launch_prefill<1, 2, 4, 4, 4, 1, std::uint64_t>(xp, codes, scales, op, tokens, n, k, padded, stream);
        return;
    }
    // The tiling with the least predicted time; the constants are a fit to 770
    // shapes (33-8192 tokens, 256-151936 rows, 64-25600 columns; each candidate
    // timed on each shape on MI355X): the choice is within 11% of the fastest
    // candidate on every one of them and 0.2% on average. The two without a K
    // split share a CU (two and four workgroups) and win where K is short, so
    // that prologue and output count (16384 rows x 256 columns, 8192 tokens:
    // 256 x 128 tiles 198 us, these 147; 100 tokens x 34816 rows x 136: the
    // fastest of the others 13.6, these 8.0).
    constexpr PrefillTiling kTilings[10] = {
        {256, 128, 1, 0.6, 7.09, 19.16, 19.16}, {128, 128, 1, 0.1, 6.30, 9.70, 9.70},   {64, 128, 1, 0.1, 4.77, 5.80, 5.80},
        {128, 128, 2, 1.5, 2.33, 15.02, 27.81}, {64, 128, 4, 0.6, 1.77, 10.98, 40.16},  {80, 64, 1, 1.6, 4.23, 3.94, 3.94},
        {64, 64, 2, 2.0, 2.67, 3.91, 6.87},     {48, 64, 2, 2.4, 1.84, 2.28, 7.21},     {32, 64, 2, 2.7, 0.91, 1.59, 5.30},
        {32, 32, 1, 1.9, 1.64, 1.32, 1.32}};
    int best = fastest_tiling(kTilings, tokens, n, k);
    // The split form reads a chunk's four scales as one 8-byte word and needs
    // one whole chunk.
    if (best >= 5 && (k < 128 || !aligned(scales, 8))) best = k < 128 ? 4 : 2;
    switch (best) {
        case 0: launch_prefill<2, 2, 2, 8, 4, 1>(xp, codes, scales, op, tokens, n, k, padded, stream); break;
        case 1: launch_prefill<1, 2, 4, 8, 4, 1>(xp, codes, scales, op, tokens, n, k, padded, stream); break;
        case 2: launch_prefill<1, 2, 4, 4, 4, 2>(xp, codes, scales, op, tokens, n, k, padded, stream); break;
        case 3: launch_prefill<1, 4, 1, 8, 2, 1>(xp, codes, scales, op, tokens, n, k, padded, stream); break;
        case 4: launch_prefill<1, 4, 1, 4, 2, 1>(xp, codes, scales, op, tokens, n, k, padded, stream); break;
        case 5: launch_split<4, 5, 4>(xp, codes, scales, op, tokens, n, k, padded, stream); break;
        case 6: launch_split<4, 4, 4>(xp, codes, scales, op, tokens, n, k, padded, stream); break;
        case 7: launch_split<4, 3, 4>(xp, codes, scales, op, tokens, n, k, padded, stream); break;
        case 8: launch_split<4, 2, 4>(xp, codes, scales, op, tokens, n, k, padded, stream); break;
        default: launch_split<8, 2, 2>(xp, codes, scales, op, tokens, n, k, padded, stream); break;
    }
}

}  // namespace vt

// Extension: the Q8 A16 projection for many tokens on fp16 matrix cores (same
// arguments as venturi_q8_head_run; fp16 activations, k % 8 == 0, any token
// count; intended for prefill, M >= 33).
extern "C" __attribute__((visibility("default"))) int venturi_q8_prefill_run(const void* x, const std::int8_t* codes,
                                                                            const __half* scales, void* out,
                                                                            int tokens, int n, int k, int padded,
                                                                            int dtype, void* stream) {
    return vt::guarded([&] {
        vt::q8_prefill_launch(x, codes, scales, out, tokens, n, k, padded, dtype, static_cast<hipStream_t>(stream));
    });
}
