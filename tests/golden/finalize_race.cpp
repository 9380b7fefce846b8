// A group whose read ends while its layer is being finalized is published exactly once.
//
//   finalize_race [layers]
//
// One thread is the transport: it stores the groups' READY words and calls the completion
// callback, once per layer, at a varying moment around the owner's finalize. Prints the layers
// that ended with a group unpublished (their consumer would wait for it until its bound).
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>
#include "leanstream/weight_manager.h"

using namespace leanstream::runtime;

namespace {

constexpr uint32_t kGroups = 2;

struct Transport {
    IOCompletionCallback callback = nullptr;
    void* arg = nullptr;
    uint32_t epoch = 0;

    static int begin(void* c, IOCompletionCallback cb, void* arg, uint32_t epoch) {
        auto& t = *static_cast<Transport*>(c);
        t.callback = cb;
        t.arg = arg;
        t.epoch = epoch;
        return 0;
    }
    static int list(void*, Span<GroupId>) { return 0; }
    static int retire(void*) { return 0; }
    static SlotId slot(void*, GroupId g) { return g; }
};

void spin(uint32_t n) {
    for (volatile uint32_t i = 0; i < n; i = i + 1) {
    }
}

// Waits for `word` to reach `l`; gives its CPU away now and then, for machines with one.
void await(const std::atomic<uint32_t>& word, uint32_t l) {
    for (uint32_t n = 1; word.load(std::memory_order_acquire) != l; ++n)
        if (n % 4096 == 0) std::this_thread::yield();
}

}  // namespace

int main(int argc, char** argv) {
    const uint32_t layers = argc > 1 ? static_cast<uint32_t>(std::atoi(argv[1])) : 1000000;
    Transport io;
    ManagerConfig mc{};
    mc.group_count = kGroups;
    mc.group_bytes = mc.staging_stride = 64;
    mc.mode = ConsumerMode::Progressive;
    mc.io_backend.context = &io;
    mc.io_backend.begin = Transport::begin;
    mc.io_backend.update = Transport::list;
    mc.io_backend.consume = Transport::list;
    mc.io_backend.retire = Transport::retire;
    mc.io_backend.ready_slot = Transport::slot;
    WeightManager manager(mc);

    GroupLayout layout[kGroups];
    SlotId cache[kGroups];
    GroupId ids[kGroups];
    for (uint32_t g = 0; g < kGroups; ++g) {
        layout[g] = {g, g, 64ull * g, 64};
        cache[g] = -1;
        ids[g] = static_cast<GroupId>(g);
    }
    alignas(128) uint32_t states[32] = {};
    alignas(128) unsigned char arena[64 * kGroups];
    ExecDesc desc[kGroups];
    uint32_t indices[kGroups];
    QueueControl control{};
    LayerStorage storage{};
    storage.layout = {layout, kGroups};
    storage.cache_slots = cache;
    storage.staging = arena;
    storage.io_states = states;
    storage.queue = {desc, indices, &control, kGroups};

    std::atomic<uint32_t> go{0}, done{0};
    std::thread transport([&] {
        uint64_t sequence = 0;
        for (uint32_t l = 1; l <= layers; ++l) {
            await(go, l);
            spin(l * 7 % 61);
            for (uint32_t g = 0; g < kGroups; ++g) {
                __atomic_store_n(states + g, kIoReady, __ATOMIC_RELEASE);
                io.callback(io.arg, IOCompletion{io.epoch, ids[g], ids[g], 0, ++sequence});
            }
            done.store(l, std::memory_order_release);
        }
    });
    uint32_t lost = 0, failed = 0;
    for (uint32_t l = 1; l <= layers; ++l) {
        for (uint32_t g = 0; g < kGroups; ++g) __atomic_store_n(states + g, kIoEmpty, __ATOMIC_RELAXED);
        failed += manager.begin_layer(0, storage) != 0;
        go.store(l, std::memory_order_release);
        spin(l * 11 % 67);
        failed += manager.finalize({ids, kGroups}) != 0;
        await(done, l);
        lost += __atomic_load_n(&control.ready_count, __ATOMIC_ACQUIRE) != kGroups;
        failed += manager.retire() != 0;
    }
    transport.join();
    std::printf("layers %u unpublished %u failed %u\n", layers, lost, failed);
    return 0;
}
