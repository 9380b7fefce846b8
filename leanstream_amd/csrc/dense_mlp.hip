// gfx950 kernels of the dense batched path of LeanStream's streaming sparse INT4 MLP (batch
// 5 .. 32, bf16 x, every active group a resident core unit): matrix cores.
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <algorithm>
#include <type_traits>
#include "mlp_args.h"
#include "mlp_launch.h"

#include "mlp_device.h"

namespace lsamd {

// ---------------------------------------------------------------------------------
// Dense batched path (batch 5 .. 32, every group a resident core unit): matrix cores.
//
// Per batch row the arithmetic is the batch-1 path's: w = fp16(q * scale) exactly, fp32
// sums of exact products, fp16 roundings of g, u, silu and h, fp32 sum of h * w_down.
// The products run on v_mfma_f32_16x16x32_f16: the dequantised weights and h are fp16
// values by definition, and bf16 x converts to fp16 exactly (8 significant bits; only
// |x| < 2^-17 rounds, by less than 2^-25), so every product is exact in fp32 and only the
// summation order differs. The 16 MFMA rows are batch rows; 17 .. 32 rows take two MFMAs a
// weight fragment.
//
// MFMA fragment layout (v_mfma_f32_16x16x32_f16, checked on gfx950): lane l holds
// A[row l % 16][k 8 (l / 16) + i] and B[k 8 (l / 16) + i][col l % 16], i < 8; result
// element i is C[4 (l / 16) + i][l % 16]. Which k a slot stands for is free as long as A and
// B agree, so each lane feeds the MFMA from its own contiguous loads.
//
// Three launches: gate/up (h rows in fp16), down projection (fp32 partial rows per split of
// the units), reduction (fixed split order, then the completion word).
// ---------------------------------------------------------------------------------
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kDenseDnWaves = 8;   // down-projection waves per workgroup: four pairs
constexpr int kDenseGuWaves = 8;   // gate/up waves per workgroup
constexpr uint32_t kDenseGuGroups = 256;   // gate/up workgroups: one a CU

__device__ __forceinline__ f32x4 mfma16(h8 a, h8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// Orders a wave's own LDS accesses across its lanes (the LDS serves a wave's accesses in
// order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// h rows as the down projection's A fragments: 16-byte piece (32-neuron half, 16 batch rows,
// lane) of lane l = row % 16 + 16 ((neuron % 32) / 8), eight neurons a piece. Rows >= batch
// are zero (cleared at bind).
__device__ __forceinline__ size_t h16_index(uint32_t dest, uint32_t n, uint32_t row) {
    return ((size_t)((2 * dest + n / 32) * 2 + row / 16) * 64 + row % 16 + 16 * (n % 32 / 8)) * 8 + n % 8;
}

// Workgroup barrier ordering LDS traffic only. __syncthreads() is a release/acquire at
// workgroup scope over all memory, so it waits for every global load of the wave still
// in flight (s_waitcnt vmcnt(0)); the prefetched loads of later units must stay in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A buffer of `bytes` bytes at a wave-uniform address: a load takes a scalar base and offset
// beside the lane's, and one past the end returns zero and reads no memory. Loads that stand for
// no work (invalid items, steps past the end) are issued with bytes = 0, so that the compiler
// can still count the loads in flight.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t wave_buffer(uint64_t address, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(address), 0, (int)bytes, 0x00027000);
}

// Eight bf16 columns of x as fp16 in dequant8's pairing: columns (0, 4, 1, 5, 2, 6, 3, 7).
__device__ __forceinline__ u32x4 x_pairs(u32x4 v) {
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t a = v[i >> 1], b = v[2 + (i >> 1)];
        const f32x2 f = {__uint_as_float(i & 1 ? a & 0xffff0000u : a << 16),
                         __uint_as_float(i & 1 ? b & 0xffff0000u : b << 16)};
        o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, h2));   // round to nearest even
    }
    return o;
}

// NT consecutive scales (2-byte aligned memory) as packed pairs.
template <int NT>
__device__ __forceinline__ void load_scales(const LS_GLOBAL uint8_t* p, uint32_t (&out)[(NT + 1) / 2]) {
    typedef uint32_t any32 __attribute__((aligned(2)));
    typedef u32x2 any64 __attribute__((aligned(2)));
    typedef u32x4 any128 __attribute__((aligned(2)));
    if constexpr (NT == 1) {
        out[0] = *reinterpret_cast<const LS_GLOBAL uint16_t*>(p);
    } else if constexpr (NT == 2) {
        out[0] = *reinterpret_cast<const LS_GLOBAL any32*>(p);
    } else if constexpr (NT == 4) {
        const u32x2 v = *reinterpret_cast<const LS_GLOBAL any64*>(p);
        out[0] = v.x;
        out[1] = v.y;
    } else {
        static_assert(NT == 8, "1, 2, 4 or 8 steps a wave");
        const u32x4 v = *reinterpret_cast<const LS_GLOBAL any128*>(p);
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = v[i];
    }
}

__device__ __forceinline__ uint32_t lane_word(uint32_t v, uint32_t lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}
__device__ __forceinline__ uint64_t lane_pointer(uint64_t v, uint32_t lane) {
    return (uint64_t)lane_word((uint32_t)(v >> 32), lane) << 32 | lane_word((uint32_t)v, lane);
}

// Gate/up. An item is eight neurons of a unit: their gate rows and their up rows are the 16
// columns of a 16x16x32 MFMA's B operand (lane l % 16: gate of neuron l % 8, then up), so a
// step of 128 columns is one 16-byte weight load a lane and one decode chain. Items of eight
// neurons spread a layer over the CUs to within an eighth of a unit.
//
// A workgroup is persistent over items wg, wg + groups, ...: KW of its eight waves split D,
// NT steps each, and a wave holds the x fragments of its columns in registers for all of its
// items (32 rows x 512 columns are 128 registers at d = 4096). x is read, converted and dealt
// to the MFMA layout once per workgroup instead of once per 32 neurons (117 MB of L2 reads at
// 4096 x 224 groups, twice the weights) by a launch of its own. The weight loads of the
// next round (two items; one at d >= 4096, whose items are four steps and more) are in flight
// while a round is computed. At the end of a round the waves' partial tiles meet in LDS in a
// fixed order, one barrier a round. Two items a round are the better up to d = 2048, one above (a
// layer at 7 and 32 rows, two items against one: 1024 columns x 128 groups 15.9 and 18.5 us
// against 16.5 and 18.6, 2048 x 128 equal, 4096 x 224 32.7 and 39.6 against 32.2 and 38.4, 8192 x
// 90 30.3 and 39.6 against 28.8 and 37.4; 16 and 17 rows alike).
//
// Where the x of 17 .. 32 rows does not fit the registers (d = 8192) a workgroup takes 16 rows
// (`halves` = 2): workgroups blk and blk + 8, on one XCD, read the same weights.
struct DenseGuParams {
    const ExecDesc* core;
    const uint16_t* x;
    uint32_t core_count, batch, groups, halves;
    MlpArgs args;
    Bounds b;
};
static_assert(offsetof(DenseGuParams, args) == 32 && offsetof(DenseGuParams, b) == 32 + sizeof(MlpArgs),
              "argument segment layout of dense_gate_up_kernel");

template <int NT, int NF, int KW>
__global__ __launch_bounds__(64 * kDenseGuWaves, NT * NF <= 2 ? 4 : 2) void dense_gate_up_kernel(
    const ExecDesc* hot_core, const uint16_t* hot_x, uint32_t hot_core_count, uint32_t hot_batch, uint32_t hot_groups,
    uint32_t hot_halves, MlpArgs args, Bounds b) {
    constexpr uint32_t D = KW * NT * 128;
    constexpr uint32_t IG = kDenseGuWaves / KW;          // items a workgroup computes at a time
    constexpr int IPB = NT < 4 ? 2 : 1, WIN = IPB * NT;  // items of a round, their steps
    constexpr int TT = NT < 4 ? NT : 4, TC = NT / TT;    // x is dealt TT steps at a time
    constexpr uint32_t PPR = 16 * TT;                    // 16-byte pieces of a row of it
    constexpr uint32_t RPI = 64 / PPR, NI = 16 / RPI;    // rows per load instruction, instructions
    constexpr uint32_t kXVecs = 16 * (PPR + 1);          // rows padded by one piece: 16 rows, 16 bank groups
    constexpr uint32_t kRedVecs = IPB * kDenseGuWaves * NF * 64;   // 16-byte vectors of a round's partial tiles
    constexpr uint32_t kVecs = kDenseGuWaves * kXVecs > 2 * kRedVecs ? kDenseGuWaves * kXVecs : 2 * kRedVecs;
    __shared__ u32x4 lds[kVecs];
    const uint32_t lane = lane_id(), w = wave_id(), kw = w % KW, ig = w / KW;
    const uint32_t q = lane >> 4, c = lane & 15;
    const uint32_t half = hot_halves > 1 ? blockIdx.x / 8u & 1u : 0u;
    const uint32_t wg = hot_halves > 1 ? blockIdx.x % 8u + 8u * (blockIdx.x / 16u) : blockIdx.x;
    const uint32_t items = 8 * hot_core_count;
    const uint32_t total = wg * IG < items ? (items / IG - wg + hot_groups - 1) / hot_groups : 0u;
    if (!total) return;
    uint32_t n = min(total, 64u);
    uint32_t item = (wg + hot_groups * min(lane, n - 1)) * IG + ig;
    ExecDesc desc = hot_core[item >> 3];
    __builtin_amdgcn_sched_barrier(0);
    // x: each load of a wave is contiguous in its rows (rows past the batch read the last one: a row
    // of A only reaches its own row of the result, which nobody reads). Behind the first weights
    // instead, x waited for them: 0.7 us more at 4096 columns x 32 rows.
    u32x4 raw[NF][TC][NI];
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int tc = 0; tc < TC; ++tc)
#pragma unroll
            for (uint32_t i = 0; i < NI; ++i) {
                const uint32_t row = min(16 * (f + half) + i * RPI + lane / PPR, hot_batch - 1);
                raw[f][tc][i] = *glb(reinterpret_cast<const u32x4*>(hot_x + (size_t)row * D + kw * (NT * 128) +
                                                                    tc * (TT * 128) + 8 * (lane % PPR)));
            }
    // A batch of up to 64 items: lane i holds the addresses of item k0 + i.
    const uint32_t row = (c & 7) * 3 + (c >> 3);
    const uint32_t vw = row * (D / 2) + kw * (NT * 64) + 16 * q;
    const uint32_t vs = (row * (D / 128) + kw * NT) * 2;
    uint32_t dest = 0, mask = 0;
    uint64_t pw = 0, ps = 0;
    u32x4 ring[WIN];
    uint32_t sring[IPB][(NT + 1) / 2];
    __amdgpu_buffer_rsrc_t wp = wave_buffer(0, 0);
    auto issue = [&](uint32_t i, int t, u32x4& dst, uint32_t (&sc)[(NT + 1) / 2]) {
        if (t == 0) {
            const uint32_t at = min(i, n - 1);
            wp = wave_buffer(lane_pointer(pw, at), i < n ? lane_word(mask, at) & (8 * 3 * D / 2) : 0u);
            // past the end: the last item's scales again
            load_scales<NT>(glb(reinterpret_cast<const uint8_t*>(lane_pointer(ps, at))) + (lane_word(mask, at) & vs), sc);
        }
        dst = __builtin_amdgcn_raw_buffer_load_b128(wp, vw, 64 * t, 0);
    };
    auto open = [&](uint32_t k0) {
        if (k0) {
            n = min(total - k0, 64u);
            item = (wg + hot_groups * (k0 + min(lane, n - 1))) * IG + ig;
            desc = hot_core[item >> 3];
        }
        __builtin_amdgcn_sched_barrier(0);
        const MlpArgs a = late_params_as<DenseGuParams>()->args;
        const Bounds bd = late_params_as<DenseGuParams>()->b;
        const Unit u = resolve(a, bd, desc, (int)D);
        const bool ok = u.ok;
        // an invalid item loads no weights, and its scales from the first words of x
        pw = reinterpret_cast<uint64_t>(u.grp + (size_t)(item & 7) * (8 * 3 * D / 2));
        ps = ok ? reinterpret_cast<uint64_t>(u.sc + (size_t)(item & 7) * (8 * 3 * (D / 128)))
                : reinterpret_cast<uint64_t>(hot_x);
        mask = ok ? ~0u : 0u;
        dest = u.dest;
        // one lane per item reports it
        if (half == 0 && kw == 0 && lane < n) {
            if (!u.ok)
                __hip_atomic_fetch_or(a.status, kStatusBadDescriptor, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            else if (!(item & 7) && a.executions)
                __hip_atomic_fetch_add(a.executions + u.dest, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
#pragma unroll
        for (int s = 0; s < WIN; ++s) issue(s / NT, s % NT, ring[s], sring[s / NT]);
        __builtin_amdgcn_sched_barrier(0);
    };
    open(0);
    // x: bf16 -> paired fp16 (dequant8's order), dealt through the wave's own LDS
    h8 xa[NF][NT][4];
    u32x4* xl = lds + w * kXVecs;
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int tc = 0; tc < TC; ++tc) {
#pragma unroll
            for (uint32_t i = 0; i < NI; ++i)
                xl[(i * RPI + lane / PPR) * (PPR + 1) + lane % PPR] = x_pairs(raw[f][tc][i]);
            wave_lds_fence();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    xa[f][tc * TT + t][j] = __builtin_bit_cast(h8, xl[c * (PPR + 1) + 16 * t + 4 * q + j]);
            wave_lds_fence();
            __builtin_amdgcn_sched_barrier(0);
        }
    uint16_t* const h16 = late_params_as<DenseGuParams>()->args.h16;
    // Sum of the waves' partial tiles of the round's items (a lane's slice: row 4 q + i of fragment f,
    // column c), h from the gate (c < 8) and up (c >= 8) lanes of each neuron.
    auto finish = [&](uint32_t base, uint32_t buffer) {
        constexpr uint32_t kSlices = IPB * NF * 4;
        const float* red = reinterpret_cast<const float*>(lds) + buffer * (kRedVecs * 4) + ig * KW * (IPB * NF * 256);
#pragma unroll
        for (uint32_t sl = 0; sl < (kSlices + KW - 1) / KW; ++sl) {
            const uint32_t slice = kw + KW * sl;
            const uint32_t k = base + slice / (NF * 4), fi = slice % (NF * 4);
            if (slice >= kSlices || k >= n) break;   // wave-uniform
            const uint32_t on = lane_word(mask, k), at = lane_word(dest, k), tile = lane_word(item & 7, k);
            float v = 0.f;
#pragma unroll
            for (uint32_t k2 = 0; k2 < KW; ++k2) v += red[k2 * (IPB * NF * 256) + slice * 64 + lane];   // fixed order
            const float r = round_half(v);
            const float up =
                __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(r), 0x128, 0xF, 0xF, false));   // row_ror:8
            const float sl1 = round_half(r / (1.0f + __expf(-r)));
            const uint32_t tk = 16 * (fi / 4 + half) + 4 * q + fi % 4;
            if (on && c < 8 && tk < hot_batch)
                h16[h16_index(at, 8 * tile + c, tk)] = __builtin_bit_cast(uint16_t, (_Float16)(sl1 * up));
        }
    };
    uint32_t rounds = 0;   // rounds computed: the partial tiles' buffer
    for (uint32_t k0 = 0;;) {
        auto round = [&](uint32_t base, auto more) {
            f32x4 acc[IPB][NF][2] = {};
#pragma unroll
            for (int m = 0; m < IPB; ++m) {
                uint32_t sc[(NT + 1) / 2];
#pragma unroll
                for (int i = 0; i < (NT + 1) / 2; ++i) sc[i] = sring[m][i];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    u32x4& word = ring[m * NT + t];
                    const uint16_t s = (uint16_t)(sc[t / 2] >> (16 * (t & 1)));
                    const h2 s2 = {half_bits(s), half_bits(s)};
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        h2 v[4];
                        dequant8(word[j], s2, v);   // columns (i, i + 4) of the word's eight
                        h8 wb;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            wb[2 * i] = v[i].x;
                            wb[2 * i + 1] = v[i].y;
                        }
#pragma unroll
                        for (int f = 0; f < NF; ++f) acc[m][f][j & 1] = mfma16(xa[f][t][j], wb, acc[m][f][j & 1]);
                    }
                    if constexpr (decltype(more)::value) issue(base + m + IPB, t, word, sring[m]);
                    __builtin_amdgcn_sched_barrier(0);   // one step's decode at a time: the x fragments fill the registers
                }
                // a last round of one item leaves the second one out
                if (!decltype(more)::value && base + m + 1 >= n) break;
            }
            // Partial tiles alternate between two buffers: this barrier ends the round's
            // computation, so every wave has read the round before last (the buffer written
            // next) and written the last one (the buffer read next).
            lds_barrier();
            float* red = reinterpret_cast<float*>(lds) + (rounds & 1) * (kRedVecs * 4) + w * (IPB * NF * 256);
#pragma unroll
            for (int m = 0; m < IPB; ++m)
#pragma unroll
                for (int f = 0; f < NF; ++f)
#pragma unroll
                    for (int i = 0; i < 4; ++i) red[((m * NF + f) * 4 + i) * 64 + lane] = acc[m][f][0][i] + acc[m][f][1][i];
            ++rounds;
            if (base) finish(base - IPB, rounds & 1);
        };
        // the last round requests nothing: a load past the end costs its issue, if no memory
        uint32_t base = 0;
        for (; base + IPB < n; base += IPB) round(base, std::true_type{});
        round(base, std::false_type{});
        lds_barrier();
        finish(base, (rounds & 1) ^ 1);
        k0 += 64;
        if (k0 >= total) return;
        open(k0);
    }
}

// Down projection. A workgroup takes 256 columns (whole 128-byte lines of the weight rows) over
// one split of the units, in steps of 32 neurons (half a unit). Its waves are four pairs: the
// pairs share the split's steps, and the two waves of a pair take 128 columns (a scale block)
// each of the same step, so a step's weight lines, h and scale lines come to the CU once. No
// wave waits for another before the end.
//
// In a step lane (q, o) = (l / 16, l % 16) loads the 4-byte word (8 columns 8 o ..) of the
// eight neuron rows 8 q ... The halves of two rows' words are joined before decoding, so a
// decoded pair is (neuron n, neuron n + 1) of one column: B fragments of 16x16x32 MFMAs whose
// column l % 16 is the tile's column 8 (l % 16) + m, m < 8, with no transposition through
// LDS (the first version's two barriers, 32 KB of LDS writes and as many reads a unit made it
// 1.5 us a unit, whatever was in flight). A step's 32 row scales are one load a wave, dealt to
// the lanes through 64 bytes of its own LDS.
//
// A step's loads are in flight while the step before it is computed; with two, three and four
// steps ahead a layer's gate/up and down took 33.4, 33.9 and 34.5 us instead of 33.1 (4096
// columns x 224 groups x 32 rows): a load costs its issue, and the ones past the end of a
// wave's few steps are wasted. The partial tiles meet in LDS in a fixed order; the split's sum
// goes to its fp32 partial rows. Twice the columns a wave (8-byte loads, half the loads a byte)
// made twice the partial tiles: equal. Against the kernel before, under the tracer: 22.1 -> 15.6 us.
template <int NF>
struct DenseDnStep {
    uint32_t q[8];   // eight rows' words
    uint32_t s;      // the scale of row l % 32
    u32x4 h[NF];     // A fragments: batch row 16 f + l % 16, neurons 8 q ..
    uint32_t ok;
};

struct DenseDnParams {
    const ExecDesc* core;
    uint32_t core_count, width, splits;
    MlpArgs args;
    Bounds b;
};
static_assert(offsetof(DenseDnParams, args) == 24 && offsetof(DenseDnParams, b) == 24 + sizeof(MlpArgs),
              "argument segment layout of dense_down_kernel");

template <int NF>
__global__ __launch_bounds__(64 * kDenseDnWaves, 2) void dense_down_kernel(const ExecDesc* hot_core,
                                                                           uint32_t hot_core_count, uint32_t hot_width,
                                                                           uint32_t hot_splits, MlpArgs args,
                                                                           Bounds b) {
    constexpr uint32_t kHalf = kDenseCols / 2, kPairs = kDenseDnWaves / 2;
    __shared__ alignas(16) float red[kDenseDnWaves][16 * NF][kHalf];
    __shared__ alignas(16) uint16_t ss[kDenseDnWaves][32];
    const uint32_t D = hot_width, splits = hot_splits;
    const uint32_t lane = lane_id(), w = wave_id(), q = lane >> 4, o = lane & 15;
    // XCD-aware order (workgroup blk runs on XCD blk % 8): consecutive splits go to consecutive
    // XCDs, so with 8, 16 or 32 splits all tiles of a split, which read the same h rows and scale
    // lines, share an L2.
    const uint32_t split = blockIdx.x % splits, tile = blockIdx.x / splits;
    const uint32_t half = w & 1, pair = w >> 1;
    const uint32_t steps = 2 * hot_core_count;   // of 32 neurons
    const uint32_t s0 = (uint32_t)((uint64_t)steps * split / splits);
    const uint32_t s1 = (uint32_t)((uint64_t)steps * (split + 1) / splits);
    const uint32_t mine = s0 + pair < s1 ? (s1 - s0 - pair + kPairs - 1) / kPairs : 0u;   // this wave's steps
    f32x4 acc[NF][8] = {};
    for (uint32_t k0 = 0; k0 < mine; k0 += 64) {   // lane i holds the addresses of step k0 + i
        const uint32_t n = min(mine - k0, 64u);
        const uint32_t my = s0 + pair + kPairs * (k0 + min(lane, n - 1));
        const ExecDesc desc = hot_core[my >> 1];
        const MlpArgs a = late_params_as<DenseDnParams>()->args;
        const Bounds bd = late_params_as<DenseDnParams>()->b;
        const Unit u = resolve(a, bd, desc, (int)D);   // an invalid descriptor is reported by the gate/up kernel
        // an invalid step loads nothing (its addresses are those of slot, row and destination 0)
        const uint32_t mask = u.ok ? ~0u : 0u;
        const uint64_t pq = reinterpret_cast<uint64_t>(u.grp) + (size_t)(32 * (my & 1) * 3 + 2) * (D / 2) +
                            tile * (kDenseCols / 2) + half * (kHalf / 2);
        const uint64_t ps = reinterpret_cast<uint64_t>(u.sc + (size_t)(32 * (my & 1) * 3 + 2) * (D / 128) + 2 * tile + half);
        const uint64_t ph = reinterpret_cast<uint64_t>(a.h16 + (size_t)(2 * u.dest + (my & 1)) * 1024);
        const uint32_t vq = 8 * q * (3 * D / 2) + 4 * o;
        const uint32_t vs = (lane & 31) * (3 * (D / 128)) * 2;
        auto issue = [&](uint32_t i, DenseDnStep<NF>& L) {
            L.ok = lane_word(mask, i);
            const __amdgpu_buffer_rsrc_t rows = wave_buffer(lane_pointer(pq, i), L.ok & (31 * (3 * D / 2) + kHalf / 2));
            const __amdgpu_buffer_rsrc_t hp = wave_buffer(lane_pointer(ph, i), L.ok & 2048u);
#pragma unroll
            for (int r = 0; r < 8; ++r) L.q[r] = __builtin_amdgcn_raw_buffer_load_b32(rows, vq, r * (3 * D / 2), 0);
            L.s = *reinterpret_cast<const LS_GLOBAL uint16_t*>(glb(reinterpret_cast<const uint8_t*>(lane_pointer(ps, i))) + vs);
#pragma unroll
            for (int f = 0; f < NF; ++f) L.h[f] = __builtin_amdgcn_raw_buffer_load_b128(hp, 16 * lane, 1024 * f, 0);
        };
        auto compute = [&](const DenseDnStep<NF>& L) {
            if (!L.ok) return;   // wave-uniform
            ss[w][lane & 31] = (uint16_t)L.s;
            wave_lds_fence();
            const u32x4 sv = *reinterpret_cast<const u32x4*>(&ss[w][8 * q]);
            wave_lds_fence();
            h8 ha[NF];
#pragma unroll
            for (int f = 0; f < NF; ++f) ha[f] = __builtin_bit_cast(h8, L.h[f]);
#pragma unroll
            for (int part = 0; part < 2; ++part) {   // columns 8 o + 4 part + k
                h2 v[4][4];                          // [row pair][k]
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    const uint32_t word = __builtin_amdgcn_perm(L.q[2 * p + 1], L.q[2 * p],
                                                                part ? 0x07060302u : 0x05040100u);
                    dequant8(word, as_h2(sv[p]), v[p]);
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    h8 wb;
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        wb[2 * p] = v[p][k].x;
                        wb[2 * p + 1] = v[p][k].y;
                    }
#pragma unroll
                    for (int f = 0; f < NF; ++f) acc[f][4 * part + k] = mfma16(ha[f], wb, acc[f][4 * part + k]);
                }
            }
        };
        DenseDnStep<NF> cur, next;
        issue(0, cur);
#pragma unroll 1
        for (uint32_t i = 1; i < n; ++i) {
            issue(i, next);
            compute(cur);
            cur = next;
        }
        compute(cur);
    }
    // Row 16 f + 4 q + i, columns 8 o + m: a lane's two float4 in the two halves of a row (a
    // wave's 16-byte accesses are then contiguous within 16 lanes).
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int part = 0; part < 2; ++part)
                *reinterpret_cast<f32x4*>(&red[w][16 * f + 4 * q + i][64 * part + 4 * o]) =
                    f32x4{acc[f][4 * part][i], acc[f][4 * part + 1][i], acc[f][4 * part + 2][i], acc[f][4 * part + 3][i]};
    __syncthreads();
    const MlpArgs a = late_params_as<DenseDnParams>()->args;
    constexpr uint32_t kQuads = kDenseCols / 4;
#pragma unroll
    for (uint32_t p = 0; p < 16 * NF * kQuads / (64 * kDenseDnWaves); ++p) {
        const uint32_t e = threadIdx.x + 64 * kDenseDnWaves * p, row = e / kQuads, j = e % kQuads;
        const uint32_t hj = j / (kHalf / 4), jj = j % (kHalf / 4);   // column half, float4 of it
        f32x4 v = {};
#pragma unroll
        for (uint32_t k = 0; k < kPairs; ++k)   // fixed order: deterministic
            v += *reinterpret_cast<const f32x4*>(&red[2 * k + hj][row][64 * (jj & 1) + 4 * (jj >> 1)]);
        if (row < a.batch)
            *reinterpret_cast<f32x4*>(a.dpart + ((size_t)split * 32 + row) * D + tile * kDenseCols + 4 * j) = v;
    }
}

// Sum of the splits in a fixed order, fp16 rounding, completion word.
// The queue of a dense launch (batch 5 .. 32) is not consumed: every group of a dense layer
// is a resident core unit. Block 0 of the reduction waits for the layer epoch (bounded) and
// raises kStatusQueueUnconsumed if the layer published queue entries, whose groups the
// output then lacks.
__device__ __forceinline__ void check_dense_queue(const MlpArgs& a, uint32_t* slot) {
    Waiter wt(a.spin_limit);
    for (;;) {
        const uint64_t te = ld_sys64(&a.control->total_count);
        if ((uint32_t)(te >> 32) == a.epoch) {
            if ((uint32_t)te) raise_status(a, slot, kStatusQueueUnconsumed);
            return;
        }
        if (ld_sys(&a.control->error)) {
            raise_status(a, slot, kStatusQueueError);
            return;
        }
        if (wt.expired()) {
            raise_status(a, slot, kStatusTimeout);
            return;
        }
        __builtin_amdgcn_s_sleep(8);
    }
}

// Completion of a dense launch: the word is stored once every column block has counted out, by one
// wave, whatever the bound on waits. The last block polls the counters, as a fused launch's mirror
// does (the blocks count out without waiting for an answer: two returning levels made the
// launch's end a round trip longer). When its bound passes first -- column blocks that wait for a
// CU behind another stream's kernel -- it leaves the launch's sequence in kSyncExit: a
// block that has counted out looks there, and the one that finds every block out stores the
// word. The poller leaves the sequence before its own last look and a block counts before its own
// (each acknowledged), so one of them sees the other; whoever takes the sequence out stores.
__device__ __forceinline__ void take_over(const MlpArgs& a, uint32_t* slot, uint32_t blocks) {
    const uint32_t lane = lane_id();
    const uint32_t want = lane < 8u ? (blocks + 7u - lane) / 8u : 0u;   // blocks b with b % 8 == lane
    const uint32_t got = lane < 8u ? ld_agent(slot + kSyncExitGroups + lane * kLine) : 0u;
    uint32_t seq = a.seq;
    if (__all(got >= want) && lane == 0 &&
        __hip_atomic_compare_exchange_strong(glb(slot + kSyncExit), &seq, 0u, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
        store_done(a);
}

__device__ __forceinline__ void await_blocks(const MlpArgs& a, uint32_t* slot, uint32_t blocks) {
    bool out = a.spin_limit != 0;
    if (out) poll_workers(a, slot, blocks, [&] { out = false; });
    if (out) {
        store_done(a);
        return;
    }
    if (lane_id() == 0) st_agent(slot + kSyncExit, a.seq);
    drain_vmem();
    take_over(a, slot, blocks);
}

struct DenseReduceParams {
    const float* dpart;
    uint32_t width, batch, dsplits;
    MlpArgs args;
};
static_assert(offsetof(DenseReduceParams, args) == 24, "argument segment layout of dense_reduce_kernel");

// The column blocks' split loads go out from the preloaded arguments; the argument block is
// read behind them.
__global__ __launch_bounds__(kThreads) void dense_reduce_kernel(const float* hot_dpart, uint32_t hot_width,
                                                                uint32_t hot_batch, uint32_t hot_dsplits,
                                                                MlpArgs args) {
    // the launch's last block (the column blocks are counted from the preloaded arguments)
    if (blockIdx.x == (hot_batch * hot_width / 4 + kThreads - 1) / kThreads) {
        const MlpArgs a = late_params_as<DenseReduceParams>()->args;
        uint32_t* slot = a.sync + (a.seq & 1) * a.slot_words;
        // The last block only clears the next launch's ring slot (its last user, the previous
        // launch, has finished: stream order) and checks the layer's queue (a read of host
        // memory), in parallel with the column blocks; this kernel runs in every dense
        // launch, with or without core units.
        uint32_t* other = a.sync + ((a.seq + 1) & 1) * a.slot_words;
        for (uint32_t i = threadIdx.x; i < ring_words_used(a); i += blockDim.x) st_agent(other + i, 0u);
        if (threadIdx.x < 64) {
            if (threadIdx.x == 0) check_dense_queue(a, slot);
            drain_vmem();   // a status bit raised there precedes the completion word
        }
        __syncthreads();   // the next ring slot is clear
        if (threadIdx.x < 64) await_blocks(a, slot, blockIdx.x);
        return;
    }
    // four consecutive columns of one row per thread (width is a multiple of 256): every
    // split's 16-byte load in flight
    const uint32_t idx = 4 * (blockIdx.x * kThreads + threadIdx.x);   // row * D + column
    const uint32_t W = hot_width;
    const LS_GLOBAL float4* parts = glb(reinterpret_cast<const float4*>(hot_dpart));
    float4 v = {0.f, 0.f, 0.f, 0.f};
    const bool mine = idx < hot_batch * W;
    if (mine) {
        const uint32_t tk = idx / W, col = idx - tk * W;
        // every split's load in flight
        float4 p[kDenseSplits];
#pragma unroll
        for (uint32_t s = 0; s < kDenseSplits; ++s)
            if (s < hot_dsplits) p[s] = parts[(((size_t)s * 32 + tk) * W + col) / 4];
#pragma unroll
        for (uint32_t s = 0; s < kDenseSplits; ++s)
            if (s < hot_dsplits) {
                v.x += p[s].x;
                v.y += p[s].y;
                v.z += p[s].z;
                v.w += p[s].w;
            }
    }
    const MlpArgs a = late_params_as<DenseReduceParams>()->args;
    uint32_t* slot = a.sync + (a.seq & 1) * a.slot_words;
    if (mine) {
        if (a.y32) *reinterpret_cast<float4*>(a.y32 + idx) = v;
        const uint32_t lo = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v.x) |
                            (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v.y) << 16;
        const uint32_t hi = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v.z) |
                            (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v.w) << 16;
        *reinterpret_cast<u32x2*>(a.y + idx) = u32x2{lo, hi};
    }
    count_out(slot);
    if (threadIdx.x < 64) {
        drain_vmem();   // counted
        if (ld_agent(slot + kSyncExit) == a.seq) take_over(a, slot, gridDim.x - 1);
    }
}

namespace {
// Gate/up kernels by width and rows: D = 128 x steps x waves an item is split over.
struct DenseGu {
    const void* fn;
    uint32_t items;    // items a workgroup computes at a time
    uint32_t halves;   // workgroups the rows of an item are split over
};
template <int NT, int NF, int KW>
DenseGu dense_gu(uint32_t halves = 1) {
    return {reinterpret_cast<const void*>(&dense_gate_up_kernel<NT, NF, KW>), (uint32_t)(kDenseGuWaves / KW), halves};
}
DenseGu dense_gate_up_for(uint32_t width, uint32_t batch) {
    const bool two = batch > 16;
    switch (width) {
        case 512: return two ? dense_gu<1, 2, 4>() : dense_gu<1, 1, 4>();
        case 1024: return two ? dense_gu<1, 2, 8>() : dense_gu<1, 1, 8>();
        case 2048: return two ? dense_gu<2, 2, 8>() : dense_gu<2, 1, 8>();
        case 4096: return two ? dense_gu<4, 2, 8>() : dense_gu<4, 1, 8>();
        case 8192: return dense_gu<8, 1, 8>(two ? 2 : 1);
        default: return {nullptr, 0, 0};
    }
}
}  // namespace

bool dense_available(int width) { return width > 0 && dense_gate_up_for((uint32_t)width, 1).fn != nullptr; }

hipError_t launch_dense(const MlpArgs& args, const Bounds& bounds, hipStream_t stream) {
    MlpArgs a = args;
    Bounds b = bounds;
    const DenseGu gu = dense_gate_up_for(a.width, a.batch);
    if (a.group_size != 64 || !gu.fn || a.batch <= kMaxBatch || a.batch > kMaxDenseBatch || !a.dsplits ||
        !a.h16 || !a.dpart)
        return hipErrorInvalidValue;
    hipError_t e = hipSuccess;
    if (a.core_count) {
        // groups of workgroups over the items; whole rows of XCDs where the batch is split
        uint32_t groups = std::min(kDenseGuGroups / gu.halves, 8 * a.core_count / gu.items);
        if (gu.halves > 1) groups = (groups + 7) / 8 * 8;
        uint32_t halves = gu.halves;
        void* gargs[] = {&a.core, &a.x, &a.core_count, &a.batch, &groups, &halves, &a, &b};
        e = hipLaunchKernel(gu.fn, dim3(groups * halves), dim3(64 * kDenseGuWaves), gargs, 0, stream);
        // One workgroup a CU, and a split for every four steps, one a wave pair (rounded up: a
        // small layer's pairs may be idle, no split is).
        const uint32_t tiles = a.width / kDenseCols;
        a.dsplits = std::min(dense_splits(a.width), (2 * a.core_count + kDenseDnWaves / 2 - 1) / (kDenseDnWaves / 2));
        void* dargs[] = {&a.core, &a.core_count, &a.width, &a.dsplits, &a, &b};
        const void* down = a.batch > 16 ? reinterpret_cast<const void*>(&dense_down_kernel<2>)
                                        : reinterpret_cast<const void*>(&dense_down_kernel<1>);
        if (e == hipSuccess)
            e = hipLaunchKernel(down, dim3(tiles * a.dsplits), dim3(64 * kDenseDnWaves), dargs, 0, stream);
    } else {
        a.dsplits = 0;   // nothing to sum: y = 0
    }
    if (e != hipSuccess) return e;
    // four columns per thread, plus one block for the ring slot and the queue check
    const float* dpart = a.dpart;
    void* rargs[] = {&dpart, &a.width, &a.batch, &a.dsplits, &a};
    return hipLaunchKernel(reinterpret_cast<const void*>(&dense_reduce_kernel),
                           dim3((a.batch * a.width / 4 + kThreads - 1) / kThreads + 1), dim3(kThreads), rargs, 0,
                           stream);
}

}  // namespace lsamd
