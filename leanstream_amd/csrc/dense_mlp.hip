// gfx950 kernels of the dense batched path of LeanStream's streaming sparse INT4 MLP (batch
// 5 .. 32, bf16 x, every active group a resident core unit): matrix cores.
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
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
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kDenseCols = 256;    // down-projection columns per workgroup: whole 128-byte weight lines
constexpr int kDenseDnWaves = kDenseCols / 32;   // 32 columns per wave
constexpr int kDensePitch = 72;    // fp16 per LDS row: 64 neurons + 8 (rows stay 16-byte aligned)
constexpr int kDenseGuWaves = 8;   // gate/up waves per workgroup, each reduces D / 8 columns
constexpr int kDensePrefetch = 6;  // units whose down-tile loads are in flight per workgroup (9 loads each)
constexpr int kDenseGuWindow = 3;  // gate/up steps (64 columns) whose weight loads a wave keeps in flight

__device__ __forceinline__ _Float16 bf16_to_f16(uint32_t bits) {
    return (_Float16)__builtin_bit_cast(float, bits << 16);
}

__device__ __forceinline__ f32x16 mfma32(h8 a, h8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
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
    const uint32_t G = a.group_size;
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
    const uint32_t hstride = a.slot_capacity * G;
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
            a.h16[(size_t)tk * hstride + u.dest * G + half * 32 + (l & 31)] =
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

// One unit's share of a down-projection workgroup's loads. Thread t covers rows
// 4 (t / 32) .. + 3 and columns 8 (t % 32) .. + 7 of the unit's 64 x 256 weight tile: one
// 4-byte load per row (a wave's 32 lanes read a row's whole 128-byte line), that row's
// scale for the columns' block, and 8 bytes of the unit's h rows (batch row t / 16,
// neurons 4 (t % 16) ..).
struct DenseDnLoad {
    uint32_t q[4], sb[4];
    u32x2 hv;
    bool ok;
};

// Branch-free, so that the compiler can count the loads in flight and wait for exactly
// one unit's: a position past the split, and an invalid descriptor, issue the same loads
// at the first word of the h rows for every lane (one line per instruction instead of a
// unit's 8 KB tile again; the h rows are not written by this kernel), with ok = false.
// h rows >= batch are zero (cleared at bind).
__device__ __forceinline__ void dense_dn_issue_desc(const MlpArgs& a, const Bounds& b, ExecDesc d, bool in, uint32_t c0,
                                                    DenseDnLoad& L) {
    const uint32_t D = a.width, G = a.group_size, t = threadIdx.x;
    const uint32_t nq = t >> 5, o = t & 31, hr = t >> 4, hp = t & 15;
    const Unit u = resolve(a, b, d, (int)D);
    L.ok = in && u.ok;   // an invalid descriptor is reported by the gate/up kernel
    const uint8_t* grp = L.ok ? u.grp : reinterpret_cast<const uint8_t*>(a.h16);
    const uint16_t* sc = L.ok ? u.sc : a.h16;
    const uint32_t col = c0 + 8 * o;
    const uint32_t on = L.ok ? 1u : 0u;   // 0: every lane reads the h rows' first word
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint32_t n = 4 * nq + r;
        L.q[r] = *reinterpret_cast<const uint32_t*>(grp + on * ((size_t)(n * 3 + 2) * (D / 2) + col / 2));
        L.sb[r] = sc[on * ((size_t)(n * 3 + 2) * (D / 128) + col / 128)];
    }
    L.hv = *reinterpret_cast<const u32x2*>(a.h16 + on * ((size_t)hr * a.slot_capacity * G + u.dest * G + 4 * hp));
}

__device__ __forceinline__ void dense_dn_issue(const MlpArgs& a, const Bounds& b, uint32_t un, uint32_t u0,
                                               uint32_t u1, uint32_t c0, DenseDnLoad& L) {
    const bool in = un < u1;
    dense_dn_issue_desc(a, b, a.core[in ? un : u0], in, c0, L);
}

// LDS position (in halves) of the 8-neuron granule gr of tile column col: rows of 64
// neurons (128 bytes, so every column starts on the same bank), granules XOR-swizzled by
// (col ^ col >> 3) & 7: eight consecutive columns (the MFMA's 16-byte reads) take eight
// different granule slots, and so do eight columns 8 apart (the 8-byte writes of one
// instruction). Swizzling by bits 3..5 alone left the reads of eight consecutive columns on
// one slot: a third more bank-conflict cycles in the down kernel (SQ_LDS_BANK_CONFLICT).
__device__ __forceinline__ uint32_t dn_tile_pos(uint32_t col, uint32_t gr) {
    return col * 64 + 8 * (gr ^ ((col ^ (col >> 3)) & 7));
}

// Down projection of 256 columns over one split of the units. Per unit the workgroup
// dequantises the 64 x 256 weight tile into LDS transposed (column-major, 8-neuron
// granules, so a lane's eight k slots are eight neurons of its column: one 16-byte LDS
// read) and stages the unit's h rows; wave w then runs four MFMAs for columns
// 32 w .. 32 w + 31. The loads of the next kDensePrefetch units are in flight while a
// unit is computed.
__global__ __launch_bounds__(64 * kDenseDnWaves) void dense_down_kernel(MlpArgs a, Bounds b) {
    __shared__ alignas(16) _Float16 wl[kDenseCols * 64];
    __shared__ alignas(16) _Float16 hl[32][kDensePitch];
    const uint32_t D = a.width;
    const uint32_t tiles = D / kDenseCols;
    // XCD-aware order: workgroup blk runs on XCD blk % 8; the tiles of a split go to one
    // XCD (kDenseSplits is a multiple of 8), so the split's h rows and down-scale lines
    // are fetched into that XCD's L2 once instead of once per XCD
    static_assert(kDenseSplits % 8 == 0, "two splits per XCD");
    const uint32_t xcd = blockIdx.x % 8u, j = blockIdx.x / 8u;
    const uint32_t split = xcd + 8u * (j / tiles), ct = j % tiles;
    const uint32_t c0 = ct * kDenseCols;
    const uint32_t per = (a.core_count + a.dsplits - 1) / a.dsplits;
    const uint32_t u0 = min(a.core_count, split * per), u1 = min(a.core_count, u0 + per);
    const uint32_t t = threadIdx.x;
    const int lane = lane_id();
    const uint32_t w = wave_id();
    const uint32_t nq = t >> 5, o = t & 31;    // weight tile: 4-row group, 8-column group
    const uint32_t hr = t >> 4, hp = t & 15;   // h tile: batch row, 4-neuron part
    f32x16 acc = {};
    DenseDnLoad buf[kDensePrefetch];
    if (u0 < u1) {
#pragma unroll
        for (int s = 0; s < kDensePrefetch; ++s) dense_dn_issue(a, b, u0 + s, u0, u1, c0, buf[s]);
        for (uint32_t base = u0; base < u1; base += kDensePrefetch) {
#pragma unroll
            for (int s = 0; s < kDensePrefetch; ++s) {
                if (buf[s].ok) {   // uniform across the workgroup
                    // dequantise the four rows (pairs (column k, column k + 4) per row)
                    h2 v[4][4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const h2 s2 = {half_bits((uint16_t)buf[s].sb[r]), half_bits((uint16_t)buf[s].sb[r])};
                        dequant8(buf[s].q[r], s2, v[r]);
                    }
                    lds_barrier();   // the previous unit's tiles are read
#pragma unroll
                    for (int c = 0; c < 8; ++c) {   // column 8 o + c: rows 4 nq .. 4 nq + 3
                        const int k = c & 3;
                        const bool hi = c >= 4;
                        const h2 r01 = {hi ? v[0][k].y : v[0][k].x, hi ? v[1][k].y : v[1][k].x};
                        const h2 r23 = {hi ? v[2][k].y : v[2][k].x, hi ? v[3][k].y : v[3][k].x};
                        const uint32_t col = 8 * o + c;
                        *reinterpret_cast<u32x2*>(wl + dn_tile_pos(col, nq >> 1) + 4 * (nq & 1)) =
                            u32x2{__builtin_bit_cast(uint32_t, r01), __builtin_bit_cast(uint32_t, r23)};
                    }
                    *reinterpret_cast<u32x2*>(&hl[hr][4 * hp]) = buf[s].hv;
                    lds_barrier();
                    const uint32_t col = 32 * w + (lane & 31);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t gr = 2 * j + (lane >> 5);
                        const h8 ha = *reinterpret_cast<const h8*>(&hl[lane & 31][8 * gr]);
                        const h8 wb = *reinterpret_cast<const h8*>(wl + dn_tile_pos(col, gr));
                        acc = mfma32(ha, wb, acc);
                    }
                }
                dense_dn_issue(a, b, base + kDensePrefetch + s, u0, u1, c0, buf[s]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const uint32_t tk = 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        if (tk < a.batch) a.dpart[((size_t)split * 32 + tk) * D + c0 + 32 * w + (lane & 31)] = acc[i];
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
        if (hot_dsplits == kDenseSplits) {
            float4 p[kDenseSplits];
#pragma unroll
            for (uint32_t s = 0; s < kDenseSplits; ++s) p[s] = parts[(((size_t)s * 32 + tk) * W + col) / 4];
#pragma unroll
            for (uint32_t s = 0; s < kDenseSplits; ++s) {
                v.x += p[s].x;
                v.y += p[s].y;
                v.z += p[s].z;
                v.w += p[s].w;
            }
        } else {
            for (uint32_t s = 0; s < hot_dsplits; ++s) {
                const float4 q = parts[(((size_t)s * 32 + tk) * W + col) / 4];
                v.x += q.x;
                v.y += q.y;
                v.z += q.z;
                v.w += q.w;
            }
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
        void* dargs[] = {&a, &b};
        if (e == hipSuccess)
            e = hipLaunchKernel(reinterpret_cast<const void*>(&dense_down_kernel),
                                dim3(a.width / kDenseCols * a.dsplits), dim3(64 * kDenseDnWaves), dargs, 0, stream);
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
