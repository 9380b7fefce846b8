// gfx950 kernels for LeanStream's streaming sparse INT4 MLP.
//
// Arithmetic (LeanStream kernels/streaming_mlp.cu:11-41, backends/triton/core.py:9-17):
//   w      = fp16( q * scale[c/128] ),  q = signed low-nibble-first INT4
//   gate   = sum_c w_gate(c) x(c)   up = sum_c w_up(c) x(c)          (fp32)
//   h      = fp16( fp16(silu(fp16(gate))) * fp16(up) )
//   y[c]   = fp16( sum over the U destination rows of sum_n h_n w_down(n, c) )  (fp32)
//
// Work decomposition (MI355X-specific). The units of a launch (descriptors, one group of
// G neurons each) are cut into wave-sized items of a few KB of weights:
//   - gate/up items: NPI neurons of one unit (about 8 KB of weights); one 64-lane wave
//     computes their gate and up rows and publishes h;
//   - down items: one 256-column tile (two scale blocks) of one unit over all G rows.
// All gate/up items come first, then the down items (unit-major). Wave w of the
// persistent grid takes items w, w + NW, w + 2 NW, ..., one in flight at a time; with
// two workgroups per CU (8 waves) nearly the whole layer is in flight at once at the
// Ministral-8B shape, and HBM delivers it front to back. A down item needs the h of its
// unit, produced by items about one round earlier, so it is normally ready by the time
// the down weights arrive. Waves of a workgroup never wait for each other on this path;
// a wave waits for h only after all of its own gate/up items.
//
// Exactness: dequantisation is exact (dequant8); products w*x are exact in fp32; only the
// fp32 summation order differs from the reference.
//
// Reduction: a down item's 128 column sums are added into packed fixed-point column
// accumulators (kAccOne in mlp_args.h). Integer addition is associative, so y does not
// depend on the order in which items finish: the output is bit-identical across consumer
// modes, publication orders and entry points. The U-th contribution of a column
// converts it to fp32 / fp16.
//
// Cross-workgroup data (h, accumulators, counters) uses agent-scope relaxed atomics,
// which compile to sc1 loads/stores that are coherent across the eight XCD L2s. An h
// word carries its launch tag in the same 64-bit word, so no fence orders it. No acquire
// or release fence is issued inside a spin loop (those expand to whole-L2 invalidate /
// write-back). Every wait is bounded by a wall-clock limit; on expiry the status word
// records a timeout and every worker leaves.
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <algorithm>
#include "mlp_args.h"
#include "mlp_launch.h"

#include "mlp_device.h"

namespace lsamd {

// One persistent worker workgroup of a launch. Its waves walk their share of the resident
// (core) units' items, then their share of the queue's (waiting for each position to be
// published when the launch started before the queue was complete) or, with claim_batch
// > 0 on the progressive path, the items of the ready positions the workgroup claims,
// which its four waves share. Every range goes through the one call of
// process_items below, so the item loop exists once in the kernel's code (one copy per
// range kind would triple the code and raise the register count).
// Item walks of the persistent kernels: plain (one item in flight per wave, in registers),
// staged (64-neuron groups at batch 1: items staged through LDS slots), packed (groups of at
// most 32 neurons at batch 1: the plain walk with down items over packs of core units).
enum Walk : int { kWalkPlain = 0, kWalkStaged = 1, kWalkPacked = 2 };

// A worker's first loads, from the preloaded arguments only (the kernel then reads its
// argument block): its role, x (one row at batch 1) and, on the staged walk, the first
// descriptor batch of the resident range.
template <int D>
struct WorkerStart {
    WaveRole role;
    XPart<D> xp;
    Prefetched first;
};

template <int D, bool CORE, bool QUEUE, int NB, int WALK>
__device__ __forceinline__ void start_worker(const uint16_t* x, const ExecDesc* core, uint32_t core_count,
                                             uint32_t grid, uint32_t shape, u32x4* xl, WorkerStart<D>& st) {
    const uint32_t W = QUEUE ? grid - 1 : grid;
    // Roles by workgroup: the first gu_wgs workgroups take the gate/up items, the others
    // the down items (one workgroup alone takes both).
    const uint32_t gu_wgs = kSplitRoles && W >= 2 ? (W + 1) / 2 : 0;
    st.role = WaveRole{blockIdx.x * kWaves + wave_id(), W * kWaves, gu_wgs * kWaves};
    const uint32_t G = shape_group(shape), batch = shape_batch(shape);
    load_x<D>(x, NB == 1 ? 1u : batch, st.xp, xl);   // the NB = 1 kernels hold one row of x
    st.first = Prefetched{0, false};
    if constexpr (CORE) {
        if constexpr (WALK == kWalkStaged)
            prefetch_core_descs<D>(core, core_count, shape_tiles(shape) ? kDnCols : 0u, st.role, st.first);
        else
            prefetch_core_descs_plain<D, NB, WALK == kWalkPacked>(core, core_count, G, batch, st.role, st.first);
    }
}

template <int D, bool FUSED, bool CORE, bool QUEUE, int NB, int WALK>
__device__ __forceinline__ void worker(const MlpArgs& a, const Bounds& b, Shared& sh, u32x4* xl, u32x4* stage,
                                       uint32_t* slot, WorkerStart<D>& st) {
    constexpr bool STAGED = WALK == kWalkStaged;
    const WaveRole role = st.role;
    const uint32_t W = QUEUE ? a.grid - 1 : a.grid;
    const uint32_t wave = wave_id();
    unsigned long long* yacc = launch_acc(a);
    XPart<D>& xp = st.xp;
    Prefetched first = st.first;
    Epoch ep = {0, 0, 0, 0};
    Pending pd;
    pd.col = -1;
    pd.n = 0;
    const uint32_t early = (QUEUE || FUSED) && lane_id() == 0 ? ld_agent(slot + kSyncEpoch) : 0u;
    if (threadIdx.x == 0) sh.xcount = 0;   // waves count themselves in once their part of x is staged
    __syncthreads();
    bool ok = true;
    enum : uint32_t { kCore, kDecide, kDone };
    uint32_t phase = CORE ? kCore : kDecide;
    for (;;) {
        uint32_t u0 = 0, u1 = 0, e = early;
        WaveRole r = role;
        if (phase == kCore) {
            u1 = a.core_count;
            phase = kDecide;
        } else if (phase == kDecide) {
            stamp(a, kStampCoreDone);
            if (!QUEUE) break;
            ok = ok && await_epoch(a, slot, ep, early);
            stamp(a, kStampEpoch);
            // One decision for the whole workgroup (claiming synchronises its waves).
            if (lane_id() == 0) sh.wpath[wave] = ok && ep.total ? ep.path : 0u;
            __syncthreads();
            uint32_t path = sh.wpath[0];
            for (int w = 1; w < kWaves; ++w)
                if (sh.wpath[w] != path) path = 0;
            path = __builtin_amdgcn_readfirstlane(path);
            // All positions published before the launch (path 2), or published while it
            // runs (path 1): every wave walks its stripe of the queue's items, waiting for
            // each item's position as needed. Pair-claiming candidates (claim_batch > 0)
            // take the positions in the reference's ranges -- static ranges of descriptor
            // indices when all were ready (persistent.py:63-69), logged here by the worker
            // that owns them; claimed ready ranges otherwise (persistent.py:71-90), taken by
            // the queue mirror -- and deal every range's items to all waves the same way.
            if (path == 2 && a.claim_batch && threadIdx.x == 0)
                for (uint32_t first = blockIdx.x * a.claim_batch; first < ep.total; first += W * a.claim_batch)
                    log_claim(a, slot, first, min(a.claim_batch, ep.total - first), kClaimStatic);
            if (path == 2 || path == 1) {
                u0 = a.core_count;
                u1 = u0 + ep.total;
                phase = kDone;
            } else {
                break;
            }
        } else {
            break;
        }
        if (u1 > u0) {
            if constexpr (STAGED) {
                ok = process_items_staged<D, FUSED>(a, sh, stage, slot, b, yacc, xp, xl, ep, e, pd, u0, u1, r, first);
                first.valid = false;   // only the resident range's first batch is prefetched
            } else {
                ok = process_items<D, FUSED, NB, WALK == kWalkPacked>(a, sh, stage, slot, b, yacc, xp, xl, ep, e, pd,
                                                                      u0, u1, r, first);
                first.valid = false;
            }
        }
    }
    stage_x<D>(xp, NB == 1 ? 1u : a.batch, xl, &sh.xcount);
    if (QUEUE) stamp(a, kStampQueueDone);
    check_pending(a, pd, FUSED && ep.known && ep.ok ? column_rows<WALK == kWalkPacked>(a, ep.total) : 0u);
    if (a.stamps) {
        drain_vmem();
        stamp(a, kStampDrained);
    }
}

// The mirror workgroup: wave 0 mirrors the queue while waves 1..3 clear what the next
// launch will use -- the other ring slot and the other accumulator buffer, both last
// used by the previous launch (finished, by stream order).
__device__ __forceinline__ void run_mirror(const MlpArgs& a, uint32_t* slot, uint64_t pre) {
    if (threadIdx.x < 64) {
        mirror_queue(a, slot, pre);
        return;
    }
    const uint32_t t = threadIdx.x - 64, n = kThreads - 64;
    uint32_t* other = a.sync + ((a.seq + 1) & 1) * a.slot_words;
    for (uint32_t i = t; i < ring_words_used(a); i += n) st_agent(other + i, 0u);
    unsigned long long* other_acc = a.yacc + (size_t)((a.seq + 1) & 1) * a.width * a.batch * kAccStride;
    for (uint32_t i = t; i < a.width * a.batch; i += n) st_agent_u64(other_acc + (size_t)i * kAccStride, 0ull);
}

// The layer's epilogue in the fused launch's last workgroup (256 threads), once every worker
// is out: epilogue_kernel's arithmetic on the same y -- each column's fp16 value formed from
// its accumulator word as the worker that completed it formed it (acc_value), read back at
// agent scope -- one batch row after the other. The inputs known before the launch (row 0's
// residual, the norm weight) are requested while the first wave still waits for the workers
// (epi_prefetch). The flags and the bell are released only when the launch raised no status
// bit and its queue carries no error (a launch whose queue was abandoned writes no rows: its
// columns are incomplete). Then the completion word.
template <int D>
struct EpiInputs {
    uint16_t res[D / kThreads];      // row 0's residual, columns t + 256 j
    uint16_t weight[D / kThreads];   // the norm weight, columns t + 256 j
};

template <int D>
__device__ __forceinline__ void epi_prefetch(const MlpArgs& a, EpiInputs<D>& in) {
    const uint32_t t = threadIdx.x;
#pragma unroll
    for (uint32_t j = 0; j < D / kThreads; ++j) {
        in.res[j] = a.residual[t + kThreads * j];
        in.weight[j] = a.norm_weight ? a.norm_weight[t + kThreads * j] : (uint16_t)0;
    }
}

// `decision` (LDS, written by thread 0 before the workgroup's barrier): 0 when the launch
// left its queue, else 1 | total << 1 with the queue's total from the mirrored epoch word.
template <int D, bool PACKED>
__device__ __forceinline__ void fused_epilogue(const MlpArgs& a, float* lanes, uint32_t decision,
                                               const EpiInputs<D>& in) {
    constexpr uint32_t PER = D / kThreads;
    static_assert(kThreads == 256 && D % kThreads == 0, "256 threads, whole columns each");
    const uint32_t t = threadIdx.x;
    // the status and queue error words (host memory): their round trip overlaps the rows
    uint32_t status = 0, error = 0;
    if (t == 0) {
        status = ld_sys(a.status);
        error = ld_sys(&a.control->error);
    }
    const bool ok = decision & 1u;
    if (ok) {
        const uint32_t U = column_rows<PACKED>(a, decision >> 1);
        const unsigned long long* acc = launch_acc(a);
        for (uint32_t r = 0; r < a.batch; ++r) {
            const size_t base = (size_t)r * D;
            unsigned long long w[PER];
            uint16_t res[PER];
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) {
                w[j] = ld_agent_u64(reinterpret_cast<const uint64_t*>(acc) + (base + t + kThreads * j) * kAccStride);
                res[j] = r ? a.residual[base + t + kThreads * j] : in.res[j];
            }
            float sum = 0.f;
            uint16_t hid[PER];
#pragma unroll
            for (uint32_t j = 0; j < PER; ++j) {
                const uint16_t y = __builtin_bit_cast(uint16_t, (_Float16)acc_value(w[j], U));
                hid[j] = epi_hidden(res[j], y, sum);
                a.hidden[base + t + kThreads * j] = hid[j];
            }
            if (a.norm_weight) {
                const float inverse = epi_inverse(sum, lanes, D, a.norm_eps);
#pragma unroll
                for (uint32_t j = 0; j < PER; ++j)
                    a.norm_out[base + t + kThreads * j] = epi_norm(hid[j], inverse, in.weight[j]);
            }
        }
    }
    // this workgroup's stores are visible at system scope before the flags; without flags the
    // completion word orders after them as after a launch's outputs (acknowledged stores)
    if (a.hidden_flag || a.norm_flag || a.bell)
        __atomic_thread_fence(__ATOMIC_RELEASE);
    else
        drain_vmem();
    __syncthreads();
    if (t == 0) {
        if (ok && !status && !error) {
            // both flags follow the rows (the release above, then the barrier); the bell follows
            // the flags: one release between them instead of one per flag
            if (a.hidden_flag) __hip_atomic_store(a.hidden_flag, a.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (a.norm_flag) __hip_atomic_store(a.norm_flag, a.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (a.bell) (void)__hip_atomic_fetch_add(a.bell, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        __hip_atomic_store(a.done, a.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}


// ---------------------------------------------------------------------------------
// Kernels. Persistent launches have gridDim.x = workers + 1; the last block mirrors.
// ---------------------------------------------------------------------------------

// LDS of a persistent workgroup beyond Shared and x: the staged kernels' item slots
// (kWaves x 2), or the other kernels' per-wave re-deal rows of the down items.
template <bool STAGED, int NB>
struct StageArea {
    static constexpr int VECS = STAGED ? 2 * kWaves * kSlotStride : kWaves * kNonStagedWaveVecs<NB>;
};

// The arguments a persistent worker needs before its first loads (x, its descriptors,
// the weight arenas, its ring slot, the grid, the launch shape) lead the kernel's argument
// list as scalars, so they can be preloaded into SGPRs at wave start
// (-amdgpu-kernarg-preload-count); the blocks of the remaining arguments are read from
// the kernel-argument segment (late_params) once x and the first descriptors are in flight.
#define LS_HOT_PARAMS                                                                                     \
    const uint16_t *hot_x, const ExecDesc *hot_core, const uint8_t *hot_cache, const uint16_t *hot_scales, \
        uint32_t *slot, uint32_t hot_core_count, uint32_t hot_seq, uint32_t hot_grid, uint32_t hot_shape,     \
        MlpArgs args, Bounds b
__device__ __forceinline__ MlpArgs with_hot(const MlpArgs& args, const uint16_t* x, const ExecDesc* core,
                                            const uint8_t* cache, const uint16_t* scales, uint32_t core_count,
                                            uint32_t seq, uint32_t grid) {
    MlpArgs a = args;
    a.x = x;
    a.core = core;
    a.cache = cache;
    a.scales = scales;
    a.core_count = core_count;
    a.seq = seq;
    a.grid = grid;
    return a;
}

// The persistent kernels' argument segment: LS_HOT_PARAMS in order, each at its natural
// alignment (the code object's argument offsets: args at 56, b right after it).
struct PersistentParams {
    const uint16_t* x;
    const ExecDesc* core;
    const uint8_t* cache;
    const uint16_t* scales;
    uint32_t* slot;
    uint32_t core_count, seq, grid, shape;
    MlpArgs args;
    Bounds b;
};
static_assert(offsetof(PersistentParams, args) == 56 && offsetof(PersistentParams, b) == 56 + sizeof(MlpArgs),
              "argument segment layout of LS_HOT_PARAMS");

__device__ __forceinline__ const PersistentParams* late_params() { return late_params_as<PersistentParams>(); }
// `slot` (this launch's ring slot, sync + (seq & 1) slot_words) is a parameter of its own.
#define LS_HOT_ARGS                                                                                   \
    with_hot(late_params()->args, hot_x, hot_core, hot_cache, hot_scales, hot_core_count, hot_seq, hot_grid)
#define LS_LATE_BOUNDS Bounds(late_params()->b)
#define LS_WORKER_START(CORE, QUEUE) \
    start_worker<D, CORE, QUEUE, NB, WALK>(hot_x, hot_core, hot_core_count, hot_grid, hot_shape, xl, st)

// Fused layer: resident (core) units, queue consumption and the compact reduction (the
// contribution completing a column writes it), one persistent launch.
template <int D, int NB, int WALK>
__global__ __launch_bounds__(kThreads, kWgPerCu) void fused_layer_kernel(LS_HOT_PARAMS) {
    static_assert(WALK == kWalkPlain || NB == 1, "the staged and packed walks serve batch 1");
    __shared__ Shared sh;
    __shared__ u32x4 xl[NB * XGeom<D>::N];
    __shared__ u32x4 stage[StageArea<WALK == kWalkStaged, NB>::VECS];
    if (blockIdx.x == hot_grid - 1) {
        const MlpArgs a = LS_HOT_ARGS;
        const uint64_t pre = threadIdx.x == 0 ? ld_sys64(&a.control->total_count) : 0;
        run_mirror(a, slot, pre);
        if (a.hidden) {   // the layer's epilogue, here once every worker is out
            EpiInputs<D> in;
            epi_prefetch<D>(a, in);
            uint32_t* decision = reinterpret_cast<uint32_t*>(stage);
            if (threadIdx.x < 64) {
                // the epoch word is final once the queue is mirrored; read while the workers finish
                const uint32_t word = threadIdx.x == 0 ? ld_agent(slot + kSyncEpoch) : 0u;
                await_workers(a, slot, a.grid - 1, false);
                if (threadIdx.x == 0) decision[0] = (word & 3u) == 1u ? 1u | (word >> 4) << 1 : 0u;
            }
            __syncthreads();
            fused_epilogue<D, WALK == kWalkPacked>(a, reinterpret_cast<float*>(stage), decision[0], in);
        } else if (threadIdx.x < 64) {
            await_workers(a, slot, a.grid - 1);
        }
    } else {
        WorkerStart<D> st;
        LS_WORKER_START(true, true);
        const MlpArgs a = LS_HOT_ARGS;
        stamp(a, kStampEntry);
        worker<D, true, true, true, NB, WALK>(a, LS_LATE_BOUNDS, sh, xl, stage, slot, st);
        stamp(a, kStampExit);
        count_out(slot);
    }
}

// Split path, stage A: resident (core) units only; no queue, no conversion.
template <int D, int NB, int WALK>
__global__ __launch_bounds__(kThreads, kWgPerCu) void stage_a_kernel(LS_HOT_PARAMS) {
    __shared__ Shared sh;
    __shared__ u32x4 xl[NB * XGeom<D>::N];
    __shared__ u32x4 stage[StageArea<WALK == kWalkStaged, NB>::VECS];
    WorkerStart<D> st;
    LS_WORKER_START(true, false);
    const MlpArgs a = LS_HOT_ARGS;
    worker<D, false, true, false, NB, WALK>(a, LS_LATE_BOUNDS, sh, xl, stage, slot, st);
}

// Split path, stage B: persistent ready-queue consumer (last block mirrors).
template <int D, int NB, int WALK>
__global__ __launch_bounds__(kThreads, kWgPerCu) void stage_b_kernel(LS_HOT_PARAMS) {
    __shared__ Shared sh;
    __shared__ u32x4 xl[NB * XGeom<D>::N];
    __shared__ u32x4 stage[StageArea<WALK == kWalkStaged, NB>::VECS];
    if (blockIdx.x == hot_grid - 1) {
        const MlpArgs a = LS_HOT_ARGS;
        const uint64_t pre = threadIdx.x == 0 ? ld_sys64(&a.control->total_count) : 0;
        run_mirror(a, slot, pre);
        return;
    }
    WorkerStart<D> st;
    LS_WORKER_START(false, true);
    const MlpArgs a = LS_HOT_ARGS;
    worker<D, false, false, true, NB, WALK>(a, LS_LATE_BOUNDS, sh, xl, stage, slot, st);
}

// Split path, compact reduction (streaming_mlp.cu:80-84): converts every column's
// accumulator to y32 / y. 256 columns per block.
template <int D>
__global__ __launch_bounds__(kThreads) void reduce_kernel(MlpArgs a) {
    const int col = blockIdx.x * kThreads + threadIdx.x;
    const unsigned long long w =
        __hip_atomic_load(launch_acc(a) + (size_t)col * kAccStride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    write_output(a, col, w, (uint32_t)(w >> 52));
    finish_launch(a, a.sync + (a.seq & 1) * a.slot_words);   // last kernel of the split launch sequence
}

// Clears both ring slots, the accumulators and the tagged h rows (bind time, after a
// failed enqueue, or when the launch sequence wraps): afterwards no stored tag can match
// a sequence number the next launches use.
__global__ void clear_sync_kernel(uint32_t* sync, uint32_t words, unsigned long long* yacc, uint32_t columns,
                                  uint64_t* hbuf, uint32_t hwords) {
    // `columns` covers both accumulator buffers, padding included
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < words; i += stride) st_agent(sync + i, 0u);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < columns; i += stride) st_agent_u64(yacc + i, 0ull);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < hwords; i += stride)
        __hip_atomic_store(hbuf + i, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------------
// Host-side launch dispatch over the compiled (width, neurons-per-item) variants.
// ---------------------------------------------------------------------------------
namespace {

struct Variant {
    int width;
    // [0] batch 1, [1] batch 2 .. kMaxBatch, [2] batch 1 with 64-neuron groups (staged),
    // [3] batch 1 with groups of at most 32 neurons (packed down items)
    const void* fused[4];
    const void* stage_a[4];
    const void* stage_b[4];
    const void* reduce;
};

// Staged kernels exist only for the widths where they fit two workgroups per CU.
template <int D, template <int, int, int> class K>
const void* staged_kernel() {
    if constexpr (staged_width(D))
        return reinterpret_cast<const void*>(K<D, 1, kWalkStaged>::fn);
    else
        return nullptr;
}

template <int D, int NB, int WALK>
struct FusedK {
    static constexpr auto fn = &fused_layer_kernel<D, NB, WALK>;
};
template <int D, int NB, int WALK>
struct StageAK {
    static constexpr auto fn = &stage_a_kernel<D, NB, WALK>;
};
template <int D, int NB, int WALK>
struct StageBK {
    static constexpr auto fn = &stage_b_kernel<D, NB, WALK>;
};

template <int D, template <int, int, int> class K>
void fill_family(const void* (&out)[4]) {
    out[0] = reinterpret_cast<const void*>(K<D, 1, kWalkPlain>::fn);
    out[1] = reinterpret_cast<const void*>(K<D, kMaxBatch, kWalkPlain>::fn);
    out[2] = staged_kernel<D, K>();
    out[3] = reinterpret_cast<const void*>(K<D, 1, kWalkPacked>::fn);
}

template <int D>
Variant make_variant() {
    Variant v{};
    v.width = D;
    fill_family<D, FusedK>(v.fused);
    fill_family<D, StageAK>(v.stage_a);
    fill_family<D, StageBK>(v.stage_b);
    v.reduce = reinterpret_cast<const void*>(&reduce_kernel<D>);
    return v;
}

// Kernel family of a launch: 0 batch 1, 1 batch 2 .. kMaxBatch, 2 staged (batch 1,
// 64-neuron groups, widths where two workgroups' slots fit a CU's LDS), 3 packed (batch 1,
// groups of at most 32 neurons).
int family(int width, int batch, int group_size, int walk = 0) {
    if (batch > 1) return 1;
    if (walk == 1) return 0;   // the plain walk serves every batch-1 shape
    if (group_size == (int)kStagedGroup && staged_width(width)) return 2;
    return group_size <= (int)kDnRows / 2 ? 3 : 0;
}

const Variant* find_variant(int width) {
    static const Variant table[] = {make_variant<256>(),  make_variant<512>(),  make_variant<1024>(),
                                    make_variant<2048>(), make_variant<4096>(), make_variant<8192>()};
    for (const Variant& v : table)
        if (v.width == width) return &v;
    return nullptr;
}

}  // namespace

bool variant_available(int width) { return find_variant(width) != nullptr; }

hipError_t resident_workers(int width, int entry_point, int batch, int group_size, int* per_cu, int walk) {
    const Variant* v = find_variant(width);
    if (!v || batch < 1 || batch > (int)kMaxBatch) return hipErrorInvalidValue;
    const int nb = family(width, batch, group_size, walk);
    const void* k = entry_point == kEntryFused ? v->fused[nb] : v->stage_b[nb];
    int n = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, kThreads, 0);
    if (e == hipSuccess && entry_point != kEntryFused) {
        int na = 0;
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&na, v->stage_a[nb], kThreads, 0);
        if (na < n) n = na;
    }
    *per_cu = std::min(n, kStampWgPerCu);
    return e;
}

hipError_t run_stage_hook(StageHook* hook, hipStream_t stream) {
    if (!hook) return hipSuccess;
    if (hook->arm) hook->rc = hook->arm(hook->context);
    return hook->b_done ? hipEventRecord(hook->b_done, stream) : hipSuccess;
}

hipError_t launch_layer(const LaunchPlan& p, const MlpArgs& args, const Bounds& bounds, hipStream_t stream,
                        StageHook* hook) {
    const Variant* v = find_variant(p.width);
    if (!v || p.workers < 1) return hipErrorInvalidValue;
    MlpArgs a = args;
    Bounds b = bounds;
    if (a.batch < 1 || a.batch > kMaxBatch) return hipErrorInvalidValue;
    const int nb = family(p.width, (int)a.batch, (int)a.group_size, p.walk);
    a.pack = nb == 3 ? kDnRows / a.group_size : 1u;   // units per down item (pack_units)
    // the persistent kernels' leading scalars (LS_HOT_PARAMS), then the argument blocks
    uint32_t grid = (uint32_t)p.workers + 1;
    uint32_t* slot = a.sync + (a.seq & 1) * a.slot_words;
    uint32_t shape = launch_shape(a.group_size, a.batch, a.dn_tile);
    void* kargs[] = {&a.x, &a.core, &a.cache, &a.scales, &slot, &a.core_count, &a.seq, &grid, &shape, &a, &b};
    if (p.entry_point == kEntryFused) {
        a.grid = grid;
        const hipError_t e = hipLaunchKernel(v->fused[nb], dim3(grid), dim3(kThreads), kargs, 0, stream);
        return e == hipSuccess ? run_stage_hook(hook, stream) : e;
    }
    hipError_t e = hipSuccess;
    if (a.core_count) {
        grid = (uint32_t)p.workers;   // stage A has no mirror workgroup
        a.grid = grid;
        e = hipLaunchKernel(v->stage_a[nb], dim3(grid), dim3(kThreads), kargs, 0, stream);
        if (e != hipSuccess) return e;
    }
    grid = (uint32_t)p.workers + 1;
    a.grid = grid;
    e = hipLaunchKernel(v->stage_b[nb], dim3(grid), dim3(kThreads), kargs, 0, stream);
    if (e == hipSuccess) e = run_stage_hook(hook, stream);
    if (e != hipSuccess) return e;
    void* rargs[] = {&a};
    return hipLaunchKernel(v->reduce, dim3(p.width * a.batch / kThreads), dim3(kThreads), rargs, 0, stream);
}

// ---------------------------------------------------------------------------------
// Epilogue: next-hidden publication (LeanStream backends/triton/reduction.py:17-28 with
// PUBLISH) and RMSNorm (examples/ministral/native/predictor_shared_input.cu:16-41), one
// workgroup per row after the layer's launch on the same stream, so every y word of the
// launch is visible to it. hidden = fp16(fp32 residual + fp32 y); RMSNorm: thread t sums
// hidden^2 over columns t, t + 256, ... in order, a halving tree over the 256 partial sums,
// inverse = 1 / sqrt(sum / width + eps) (IEEE square root and division), out =
// fp16(weight * fp16(hidden * inverse)). Products and sums are not contracted into fused
// multiply-adds, so the result is the oracle's bit for bit. The last row's workgroup to
// finish publishes the flags after a system-scope release: hidden_flag and norm_flag, then
// (released after them) bell += 1 -- unless the layer failed: its launch raised a status bit (a
// bounded wait expired, a descriptor or a value was rejected) or its queue carries an error
// (the runtime cancelled the layer; the launch left early). Then y is not the layer's output:
// the rows are written but nothing announces them.
// ---------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void epilogue_kernel(EpilogueArgs e) {
    __shared__ float lanes[256];
    __shared__ uint32_t last;
    const uint32_t t = threadIdx.x, row = blockIdx.x;
    const uint16_t* y = e.y + (size_t)row * e.width;
    const uint16_t* res = e.residual + (size_t)row * e.width;
    uint16_t* hid = e.hidden + (size_t)row * e.width;
    float sum = 0.f;
    for (uint32_t i = t; i < e.width; i += 256) hid[i] = epi_hidden(res[i], y[i], sum);
    if (e.norm_weight) {
        const float inverse = epi_inverse(sum, lanes, e.width, e.eps);
        uint16_t* out = e.norm_out + (size_t)row * e.width;
        for (uint32_t i = t; i < e.width; i += 256) out[i] = epi_norm(hid[i], inverse, e.norm_weight[i]);
    }
    if (!e.hidden_flag && !e.norm_flag && !e.bell) return;
    // this workgroup's stores are visible at system scope before it counts itself in
    __atomic_thread_fence(__ATOMIC_RELEASE);
    __syncthreads();
    if (t == 0) {
        const uint32_t before = __hip_atomic_fetch_add(e.arrivals, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_SYSTEM);
        last = before == e.rows - 1;
        if (last) {
            __hip_atomic_store(e.arrivals, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            // the launch before this one on the stream has finished: its status bits are final
            if (__hip_atomic_load(e.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) ||
                (e.queue_error && __hip_atomic_load(e.queue_error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM)))
                return;
            // one release for both flags (every row acquired above), one between them and the bell
            __atomic_thread_fence(__ATOMIC_RELEASE);
            if (e.hidden_flag) __hip_atomic_store(e.hidden_flag, e.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (e.norm_flag) __hip_atomic_store(e.norm_flag, e.epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            if (e.bell) (void)__hip_atomic_fetch_add(e.bell, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

hipError_t launch_epilogue(const EpilogueArgs& args, hipStream_t stream) {
    EpilogueArgs e = args;
    if (!e.y || !e.residual || !e.hidden || !e.rows || !e.width || (e.norm_weight && !e.norm_out) || !e.arrivals ||
        !e.status)
        return hipErrorInvalidValue;
    void* kargs[] = {&e};
    return hipLaunchKernel(reinterpret_cast<const void*>(&epilogue_kernel), dim3(e.rows), dim3(256), kargs, 0, stream);
}

hipError_t clear_sync(uint32_t* sync, uint32_t words, unsigned long long* yacc, uint32_t columns, uint64_t* hbuf,
                      uint32_t hwords, hipStream_t stream) {
    const uint32_t most = words > hwords ? words : hwords;
    uint32_t grid = (most + kThreads - 1) / kThreads;
    if (grid > 1024) grid = 1024;
    if (!grid) grid = 1;
    void* kargs[] = {&sync, &words, &yacc, &columns, &hbuf, &hwords};
    return hipLaunchKernel(reinterpret_cast<const void*>(&clear_sync_kernel), dim3(grid), dim3(kThreads), kargs, 0,
                           stream);
}

}  // namespace lsamd
