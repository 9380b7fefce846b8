// gfx950 kernels of the dense batched path of LeanStream's streaming sparse INT4 MLP (batch
// 5 .. 32, bf16 x, every active group a resident core unit): matrix cores.
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <algorithm>
#include "mlp_args.h"
#include "mlp_launch.h"

#include "mlp_device.h"

namespace lsamd {

// ---------------------------------------------------------------------------------
// Dense batched path (batch 5 .. 32, every group a resident core unit): matrix cores.
//
// Per batch row the arithmetic is the batch-1 path's: w = fp16(q * scale) exactly, fp32
// sums of exact products, fp16 roundings of g, u, silu and h, fp32 sum of h * w_down.
// The products run on v_mfma_f32_32x32x16_f16: the dequantised weights and h are fp16
// values by definition, and bf16 x converts to fp16 exactly (8 significant bits; only
// |x| < 2^-17 rounds, by less than 2^-25), so every product is exact in fp32 and only the
// summation order differs. The 32 MFMA rows are the batch rows (rows >= batch are zero).
//
// MFMA fragment layout (v_mfma_f32_32x32x16_f16, checked on gfx950): lane l holds
// A[row l % 32][k 8 (l / 32) + i] and B[k 8 (l / 32) + i][col l % 32], i < 8; result
// element i is C[8 (i / 4) + 4 (l / 32) + i % 4][l % 32]. Which k a slot stands for is
// free as long as A and B agree, so each lane feeds the MFMA from its own contiguous loads.
//
// Four launches: x conversion (bf16 -> paired fp16, once per layer), gate/up (h rows in
// fp16), down projection (fp32 partial rows per split of the units), reduction (fixed
// split order, then the completion word).
// ---------------------------------------------------------------------------------
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kDenseCols = 128;    // down-projection columns per workgroup: one scale block
constexpr int kDenseDnWaves = 8;   // down-projection waves per workgroup, sharing a split's steps
constexpr int kDenseDnWindow = 4;  // down-projection steps (32 neurons) whose loads a wave keeps in flight
constexpr uint32_t kDenseDnGroups = 256;   // down-projection workgroups: one a CU
constexpr int kDenseGuWaves = 8;   // gate/up waves per workgroup, each reduces D / 8 columns
constexpr int kDenseGuWindow = 3;  // gate/up steps (64 columns) whose weight loads a wave keeps in flight

__device__ __forceinline__ _Float16 bf16_to_f16(uint32_t bits) {
    return (_Float16)__builtin_bit_cast(float, bits << 16);
}

__device__ __forceinline__ f32x16 mfma32(h8 a, h8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

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

// x (bf16 [batch][D]) -> x16: fp16 MFMA A fragments in dequant8's pairing. Within each
// 8-column group the slots hold columns (0, 4, 1, 5, 2, 6, 3, 7), so one 16-byte piece
// is the A fragment matching a dequantised weight word. The pieces are stored in the
// order the gate/up waves load them: fragment f = 4 (c / 64) + (c % 32) / 8 holds, for
// lane l, row l % 32 and columns 64 (c / 64) + 32 (l / 32) + 8 ((c % 32) / 8) .. + 7 at
// byte 1024 f + 16 l, so every x load of a wave reads one contiguous kilobyte. Rows >=
// batch are zero. Once per layer, shared by every gate/up workgroup.
__device__ __forceinline__ uint32_t x16_piece(uint32_t row, uint32_t c) {   // 16-byte piece index
    const uint32_t f = 4 * (c / 64) + (c % 32) / 8, l = row + 32 * ((c % 64) / 32);
    return 64 * f + l;
}

// Its arguments are scalars preloaded into SGPRs: the load goes out at once.
__global__ __launch_bounds__(kThreads) void dense_x_kernel(const uint16_t* x, uint16_t* x16, uint32_t width,
                                                           uint32_t batch) {
    const uint32_t D = width, groups = D / 8;
    const uint32_t idx = blockIdx.x * kThreads + threadIdx.x;   // row * groups + group
    const uint32_t row = idx / groups, grp = idx - row * groups;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (row < batch) v = *glb(reinterpret_cast<const u32x4*>(x + (size_t)row * D + 8 * grp));
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    h8 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        o[2 * i] = bf16_to_f16((w[i >> 1] >> (16 * (i & 1))) & 0xffffu);
        o[2 * i + 1] = bf16_to_f16((w[(i + 4) >> 1] >> (16 * (i & 1))) & 0xffffu);
    }
    glb(reinterpret_cast<h8*>(x16))[x16_piece(row, 8 * grp)] = o;
}

// Gate/up of one 32-neuron half of one unit for all batch rows. Wave w reduces the
// eighth [w D/8, (w+1) D/8) of the input in NI steps of 64 columns; the eight partial
// tiles meet in LDS. Lane l (neuron 32 half + l % 32, row l % 32 of x) takes 32
// consecutive columns per step: 16 bytes of each weight row and 64 bytes of x16. Up to
// d = 4096 the kernel stays within 128 registers (four waves per SIMD: two workgroups per
// CU, so the whole layer's workgroups are resident at once) with the weights of
// kDenseGuWindow steps in flight per wave.
// The dense kernels' argument segments (each parameter at its natural alignment): the
// leading scalars are preloaded into SGPRs, the blocks are read late (late_params_as).
struct DenseGuParams {
    const ExecDesc* core;
    const uint16_t* x16;
    MlpArgs args;
    Bounds b;
};
static_assert(offsetof(DenseGuParams, args) == 16 && offsetof(DenseGuParams, b) == 16 + sizeof(MlpArgs),
              "argument segment layout of dense_gate_up_kernel");

// The unit's descriptor and the first x16 steps go out from the preloaded arguments; the
// argument blocks are read behind them.
template <int NI>
__global__ __launch_bounds__(64 * kDenseGuWaves, NI <= 8 ? 4 : 2) void dense_gate_up_kernel(
    const ExecDesc* hot_core, const uint16_t* hot_x16, MlpArgs args, Bounds b) {
    __shared__ float red[kDenseGuWaves / 2][2][16][64];   // 32 KB: two workgroups per CU fit
    constexpr uint32_t D = NI * 64 * kDenseGuWaves;
    constexpr uint32_t kq = D / kDenseGuWaves;
    const uint32_t unit = blockIdx.x >> 1, half = blockIdx.x & 1;
    const ExecDesc desc = hot_core[unit];
    const int lane = lane_id();
    const uint32_t w = wave_id();
    const uint32_t n = half * 32 + (lane & 31), hh = lane >> 5, row = lane & 31;
    // x16 of step t (four 16-byte fragments per lane, each wave-contiguous) is loaded two
    // steps ahead, from a ring of three; steps 0 and 1 go out before the weights. Loads
    // complete in issue order, so each step waits only for what it uses.
    const LS_GLOBAL u32x4* xf = glb(reinterpret_cast<const u32x4*>(hot_x16));
    u32x4 xq[3][4];
    auto issue_x = [&](int t, u32x4 (&dst)[4]) {
        const uint32_t k0 = w * kq + 64 * t + 32 * hh;
#pragma unroll
        for (int j = 0; j < 4; ++j) dst[j] = xf[x16_piece(row, k0 + 8 * j)];
    };
    issue_x(0, xq[0]);
    if (NI > 1) issue_x(1, xq[1]);
    const MlpArgs a = late_params_as<DenseGuParams>()->args;
    const Bounds bd = late_params_as<DenseGuParams>()->b;
    const Unit u = resolve(a, bd, desc, (int)D);
    f32x16 cg = {}, cu = {};
    if (u.ok) {
        const uint8_t* wg = u.grp + (size_t)(n * 3) * (D / 2);
        const uint8_t* wu = wg + D / 2;
        const uint16_t* sg = u.sc + (size_t)(n * 3) * (D / 128);
        const uint16_t* su = sg + D / 128;
        // The weights of WIN steps are in flight: step t's pieces go out into the slot
        // step t - WIN has just been computed from.
        constexpr int WIN = NI < kDenseGuWindow ? NI : kDenseGuWindow;
        u32x4 qg[WIN], qu[WIN];
        auto issue_w = [&](int t) {
            const uint32_t k0 = w * kq + 64 * t + 32 * hh;
            qg[t % WIN] = ld_cached16(wg + k0 / 2);   // a row's 128-byte line serves four steps
            qu[t % WIN] = ld_cached16(wu + k0 / 2);
        };
#pragma unroll
        for (int t = 0; t < WIN; ++t) issue_w(t);
        // The wave's K range covers SB consecutive scale blocks of each row (step t uses
        // block t / 2): one 8-byte load per projection row where SB is a multiple of 4.
        constexpr int SB = NI >= 2 ? NI / 2 : 1;
        uint32_t sgv[SB], suv[SB];
        const uint32_t b0 = NI >= 2 ? w * SB : w / 2;
        if constexpr (SB % 4 == 0) {
#pragma unroll
            for (int i = 0; i < SB; i += 4) {
                const u32x2 gv = *reinterpret_cast<const u32x2*>(sg + b0 + i);
                const u32x2 uv = *reinterpret_cast<const u32x2*>(su + b0 + i);
                sgv[i] = gv.x & 0xffffu; sgv[i + 1] = gv.x >> 16; sgv[i + 2] = gv.y & 0xffffu; sgv[i + 3] = gv.y >> 16;
                suv[i] = uv.x & 0xffffu; suv[i + 1] = uv.x >> 16; suv[i + 2] = uv.y & 0xffffu; suv[i + 3] = uv.y >> 16;
            }
        } else {
#pragma unroll
            for (int i = 0; i < SB; ++i) {
                sgv[i] = sg[b0 + i];
                suv[i] = su[b0 + i];
            }
        }
        // keep every load above ahead of the first MFMA (the scheduler would otherwise
        // sink them next to their uses, leaving two or three in flight per wave)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NI; ++t) {
            if (t + 2 < NI) issue_x(t + 2, xq[(t + 2) % 3]);
            __builtin_amdgcn_sched_barrier(0);
            const int sb = NI >= 2 ? t / 2 : 0;   // constant after unrolling
            const h2 sg2 = {half_bits((uint16_t)sgv[sb]), half_bits((uint16_t)sgv[sb])};
            const h2 su2 = {half_bits((uint16_t)suv[sb]), half_bits((uint16_t)suv[sb])};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const h8 xa = __builtin_bit_cast(h8, xq[t % 3][j]);   // paired (dense_x_kernel)
                h2 wgv[4], wuv[4];
                dequant8(qg[t % WIN][j], sg2, wgv);   // (column 8 j + i, column 8 j + i + 4)
                dequant8(qu[t % WIN][j], su2, wuv);
                h8 bg, bu;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    bg[2 * i] = wgv[i].x;
                    bg[2 * i + 1] = wgv[i].y;
                    bu[2 * i] = wuv[i].x;
                    bu[2 * i + 1] = wuv[i].y;
                }
                cg = mfma32(xa, bg, cg);
                cu = mfma32(xa, bu, cu);
            }
            if (t + WIN < NI) issue_w(t + WIN);
        }
    }
    // Fixed-order sum of the eight partial tiles: wave w + 4 into wave w, then waves 0..3.
    constexpr uint32_t HW = kDenseGuWaves / 2;
    if (w >= HW) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            red[w - HW][0][i][lane] = cg[i];
            red[w - HW][1][i][lane] = cu[i];
        }
    }
    __syncthreads();
    if (w < HW) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            red[w][0][i][lane] += cg[i];
            red[w][1][i][lane] += cu[i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 1024 / (64 * kDenseGuWaves); ++r) {
        const uint32_t e = threadIdx.x + 64 * kDenseGuWaves * r, i = e >> 6, l = e & 63;
        float gsum = 0.f, usum = 0.f;
#pragma unroll
        for (int v = 0; v < (int)HW; ++v) {   // fixed order: deterministic
            gsum += red[v][0][i][l];
            usum += red[v][1][i][l];
        }
        const uint32_t tk = 8 * (i >> 2) + 4 * (l >> 5) + (i & 3);
        if (u.ok && tk < a.batch) {
            const float g = round_half(gsum);
            const float up = round_half(usum);
            const float sl = round_half(g / (1.0f + __expf(-g)));
            a.h16[h16_index(u.dest, half * 32 + (l & 31), tk)] =
                __builtin_bit_cast(uint16_t, (_Float16)(sl * up));
        }
    }
    if (threadIdx.x == 0) {
        if (!u.ok) {
            __hip_atomic_fetch_or(a.status, kStatusBadDescriptor, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        } else if (half == 0 && a.executions) {
            __hip_atomic_fetch_add(a.executions + u.dest, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// Down projection. A workgroup takes the 128 columns (64 bytes of every weight row) of one
// column tile over one split of the units; its eight waves share the split in steps of 32
// neurons (half a unit), each step a wave's own from its loads to its matrix instructions, so
// no wave waits for another before the end.
//
// In a step lane (q, o) = (l / 16, l % 16) loads the 4-byte word (8 columns 8 o ..) of the
// eight neuron rows 8 q ... The halves of two rows' words are joined before decoding, so a
// decoded pair is (neuron n, neuron n + 1) of one column: B fragments of 16x16x32 MFMAs whose
// column l % 16 is the tile's column 8 (l % 16) + m, m < 8, with no transposition through
// LDS (the first version's two barriers, 32 KB of LDS writes and as many reads a unit made it
// 1.5 us a unit, whatever was in flight). A step's 32 row scales (a tile is one scale block)
// are one load a wave, dealt to the lanes through 64 bytes of its own LDS.
//
// The loads of kDenseDnWindow steps are in flight per wave. The eight partial tiles meet in LDS
// in a fixed order; the split's sum goes to its fp32 partial rows.
template <int NF>
struct DenseDnStep {
    uint32_t q[8];      // eight rows' words
    uint32_t s;         // the scale of row l % 32
    u32x4 h[NF];        // A fragments: batch row 16 f + l % 16, neurons 8 q ..
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

__device__ __forceinline__ uint32_t lane_word(uint32_t v, uint32_t lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}
__device__ __forceinline__ uint64_t lane_pointer(uint64_t v, uint32_t lane) {
    return (uint64_t)lane_word((uint32_t)(v >> 32), lane) << 32 | lane_word((uint32_t)v, lane);
}

template <int NF>
__global__ __launch_bounds__(64 * kDenseDnWaves, 2) void dense_down_kernel(const ExecDesc* hot_core,
                                                                           uint32_t hot_core_count, uint32_t hot_width,
                                                                           uint32_t hot_splits, MlpArgs args,
                                                                           Bounds b) {
    __shared__ alignas(16) float red[kDenseDnWaves][16 * NF][kDenseCols];
    __shared__ alignas(16) uint16_t ss[kDenseDnWaves][32];
    const uint32_t D = hot_width, splits = hot_splits;
    const uint32_t lane = lane_id(), w = wave_id(), q = lane >> 4, o = lane & 15;
    // XCD-aware order (workgroup blk runs on XCD blk % 8): the two tiles that share the
    // 128-byte lines of a weight row are neighbours on one XCD, and so, where the splits are a
    // multiple of 8, are all tiles of a split, which read the same h rows.
    const uint32_t combo = blockIdx.x % 8u + 8u * (blockIdx.x / 16u);
    const uint32_t split = combo % splits, tile = 2u * (combo / splits) + (blockIdx.x / 8u & 1u);
    if (tile >= D / kDenseCols) return;   // the grid is rounded up to whole XCD rows
    const uint32_t steps = 2 * hot_core_count;   // of 32 neurons
    const uint32_t s0 = (uint32_t)((uint64_t)steps * split / splits);
    const uint32_t s1 = (uint32_t)((uint64_t)steps * (split + 1) / splits);
    const uint32_t mine = s0 + w < s1 ? (s1 - s0 - w + kDenseDnWaves - 1) / kDenseDnWaves : 0u;   // this wave's steps
    f32x4 acc[NF][8] = {};
    for (uint32_t k0 = 0; k0 < mine; k0 += 64) {   // lane i holds the addresses of step k0 + i
        const uint32_t n = min(mine - k0, 64u);
        const uint32_t my = s0 + w + kDenseDnWaves * (k0 + min(lane, n - 1));
        const ExecDesc desc = hot_core[my >> 1];
        const MlpArgs a = late_params_as<DenseDnParams>()->args;
        const Bounds bd = late_params_as<DenseDnParams>()->b;
        const Unit u = resolve(a, bd, desc, (int)D);   // an invalid descriptor is reported by the gate/up kernel
        const bool ok = u.ok && lane < n;
        // steps past the end and invalid ones load one word of the h rows in every lane
        const uint64_t pq = reinterpret_cast<uint64_t>(
            ok ? u.grp + ((size_t)(32 * (my & 1) * 3 + 2) * (D / 2) + tile * (kDenseCols / 2))
               : reinterpret_cast<const uint8_t*>(a.h16));
        const uint64_t ps = reinterpret_cast<uint64_t>(
            ok ? u.sc + ((size_t)(32 * (my & 1) * 3 + 2) * (D / 128) + tile) : a.h16);
        const uint64_t ph = reinterpret_cast<uint64_t>(a.h16 + (ok ? (size_t)(2 * u.dest + (my & 1)) * 1024 : 0));
        const uint32_t mask = ok ? ~0u : 0u;
        const uint32_t vq = 8 * q * (3 * D / 2) + 4 * o;
        const uint32_t vs = (lane & 31) * (3 * (D / 128)) * 2;
        auto issue = [&](uint32_t i, DenseDnStep<NF>& L) {
            const uint32_t at = min(i, 63u);
            const uint32_t on = i < n ? lane_word(mask, at) : 0u;
            const auto* rows = glb(reinterpret_cast<const uint8_t*>(lane_pointer(pq, at)));
            const auto* sc = glb(reinterpret_cast<const uint8_t*>(lane_pointer(ps, at)));
            const auto* hp = glb(reinterpret_cast<const u32x4*>(lane_pointer(ph, at)));
            const uint32_t step = on & (3 * D / 2), vo = on & vq;
#pragma unroll
            for (int r = 0; r < 8; ++r) L.q[r] = *reinterpret_cast<const LS_GLOBAL uint32_t*>(rows + r * step + vo);
            L.s = *reinterpret_cast<const LS_GLOBAL uint16_t*>(sc + (on & vs));
#pragma unroll
            for (int f = 0; f < NF; ++f) L.h[f] = hp[on & (64 * f + lane)];
            L.ok = on;
        };
        DenseDnStep<NF> ring[kDenseDnWindow];
#pragma unroll
        for (int s = 0; s < kDenseDnWindow; ++s) issue(s, ring[s]);
        for (uint32_t base = 0; base < n; base += kDenseDnWindow) {
#pragma unroll
            for (int s = 0; s < kDenseDnWindow; ++s) {
                DenseDnStep<NF>& L = ring[s];
                if (L.ok) {   // wave-uniform
                    ss[w][lane & 31] = (uint16_t)L.s;
                    wave_lds_fence();
                    const u32x4 sv = *reinterpret_cast<const u32x4*>(&ss[w][8 * q]);
                    wave_lds_fence();
                    h8 ha[NF];
#pragma unroll
                    for (int f = 0; f < NF; ++f) ha[f] = __builtin_bit_cast(h8, L.h[f]);
#pragma unroll
                    for (int half = 0; half < 2; ++half) {   // columns 8 o + 4 half + k
                        h2 v[4][4];                          // [row pair][k]
#pragma unroll
                        for (int p = 0; p < 4; ++p) {
                            const uint32_t word = __builtin_amdgcn_perm(L.q[2 * p + 1], L.q[2 * p],
                                                                        half ? 0x07060302u : 0x05040100u);
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
                            for (int f = 0; f < NF; ++f) acc[f][4 * half + k] = mfma16(ha[f], wb, acc[f][4 * half + k]);
                        }
                    }
                }
                issue(base + kDenseDnWindow + s, L);
            }
        }
    }
    // Row 16 f + 4 q + i, columns 8 o + m: the two float4 of a lane in the two halves of a row
    // (a wave's 16-byte accesses are then contiguous within 16 lanes).
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float* row = red[w][16 * f + 4 * q + i];
            *reinterpret_cast<f32x4*>(row + 4 * o) = f32x4{acc[f][0][i], acc[f][1][i], acc[f][2][i], acc[f][3][i]};
            *reinterpret_cast<f32x4*>(row + 64 + 4 * o) = f32x4{acc[f][4][i], acc[f][5][i], acc[f][6][i], acc[f][7][i]};
        }
    __syncthreads();
    const MlpArgs a = late_params_as<DenseDnParams>()->args;
    constexpr uint32_t kQuads = kDenseCols / 4;
#pragma unroll
    for (uint32_t p = 0; p < 16 * NF * kQuads / (64 * kDenseDnWaves); ++p) {
        const uint32_t e = threadIdx.x + 64 * kDenseDnWaves * p, row = e / kQuads, j = e % kQuads;
        f32x4 v = {};
#pragma unroll
        for (int k = 0; k < kDenseDnWaves; ++k)   // fixed order: deterministic
            v += *reinterpret_cast<const f32x4*>(&red[k][row][64 * (j & 1) + 4 * (j >> 1)]);
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
        if (threadIdx.x == 0) check_dense_queue(a, slot);
        finish_launch(a, slot);
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
    finish_launch(a, slot);
}

namespace {
const void* dense_gate_up_for(uint32_t width) {
    switch (width) {
        case 512: return reinterpret_cast<const void*>(&dense_gate_up_kernel<1>);
        case 1024: return reinterpret_cast<const void*>(&dense_gate_up_kernel<2>);
        case 2048: return reinterpret_cast<const void*>(&dense_gate_up_kernel<4>);
        case 4096: return reinterpret_cast<const void*>(&dense_gate_up_kernel<8>);
        case 8192: return reinterpret_cast<const void*>(&dense_gate_up_kernel<16>);
        default: return nullptr;
    }
}
}  // namespace

bool dense_available(int width) { return width > 0 && dense_gate_up_for((uint32_t)width) != nullptr; }

hipError_t launch_dense(const MlpArgs& args, const Bounds& bounds, hipStream_t stream) {
    MlpArgs a = args;
    Bounds b = bounds;
    const void* gate_up = dense_gate_up_for(a.width);
    if (a.group_size != 64 || !gate_up || a.batch <= kMaxBatch || a.batch > kMaxDenseBatch || !a.dsplits ||
        !a.h16 || !a.dpart || !a.x16)
        return hipErrorInvalidValue;
    hipError_t e = hipSuccess;
    if (a.core_count) {
        uint16_t* x16 = a.x16;
        void* xargs[] = {&a.x, &x16, &a.width, &a.batch};
        e = hipLaunchKernel(reinterpret_cast<const void*>(&dense_x_kernel), dim3(32 * a.width / 8 / kThreads),
                            dim3(kThreads), xargs, 0, stream);
        const uint16_t* cx16 = a.x16;
        void* gargs[] = {&a.core, &cx16, &a, &b};
        if (e == hipSuccess)
            e = hipLaunchKernel(gate_up, dim3(2 * a.core_count), dim3(64 * kDenseGuWaves), gargs, 0, stream);
        // One workgroup a CU, and no more splits than leave each of its waves a step.
        const uint32_t tiles = a.width / kDenseCols;
        a.dsplits = std::min({kDenseSplits, std::max(1u, kDenseDnGroups / tiles),
                              (2 * a.core_count + kDenseDnWaves - 1) / kDenseDnWaves});
        const uint32_t combos = a.dsplits * (tiles / 2);
        void* dargs[] = {&a.core, &a.core_count, &a.width, &a.dsplits, &a, &b};
        const void* down = a.batch > 16 ? reinterpret_cast<const void*>(&dense_down_kernel<2>)
                                        : reinterpret_cast<const void*>(&dense_down_kernel<1>);
        if (e == hipSuccess)
            e = hipLaunchKernel(down, dim3((combos + 7) / 8 * 16), dim3(64 * kDenseDnWaves), dargs, 0, stream);
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
