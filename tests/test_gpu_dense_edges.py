"""Dense batched path (batch 5 .. 32) and the d = 8192 matrix-core products at the sizes where
their splits can go wrong, against the CPU oracle (relative L2 <= 1e-3, max-abs <= 2e-2 of the
fp32 output, as for the other widths: fp16 roundings of g, u, silu and h that a sum in another
order moves by a unit in the last place).

Dense: gate/up items of 8 neurons and their rounds (one unit; fewer items than workgroups; more than
64 items a workgroup or down steps a wave, which are taken in batches of 64), 16 and 17 batch rows
(one and two MFMA row fragments; at d = 8192 the second 16 rows go to workgroups of their own),
every width's split of the columns over waves, and down splits with idle waves. d = 8192 at batch
1 .. 4: group sizes of every walk, and every row of a batch against a launch of that row alone.
"""
import time

import numpy as np
import pytest

import oracle
from leanstream_amd.backend import MODE_PROGRESSIVE, NativeBackend, ReadyQueue
from leanstream_amd.workload import DeviceLayer

from test_gpu_widths import check_rows, config, sync_and_check_status

pytestmark = pytest.mark.gpu

REL_L2, MAX_ABS = 1e-3, 2e-2   # max-abs of outputs of root mean square up to 1; in proportion beyond
STATUS_BAD_DESCRIPTOR = 4

CASES = [(512, 5, 1), (512, 17, 3), (512, 16, 37),             # two items a workgroup at a time
         (1024, 16, 1), (1024, 17, 33), (1024, 5, 2049),       # more than 64 items a workgroup, two a round
         (2048, 7, 5), (2048, 16, 67), (2048, 17, 3),
         (4096, 6, 1), (4096, 16, 9), (4096, 17, 33), (4096, 31, 40),
         (8192, 16, 2), (8192, 17, 1), (8192, 32, 21),
         (8192, 17, 1100)]   # more than 64 items a workgroup, one a round, and more than 64 steps a down wave


def dense(torch, d, batch, units, bad=(), row=None, table=None):
    """A core-only launch over random groups; returns (y32, per-row oracle inputs, status). With
    `row`, a launch of that row of the batch alone; `table`: an offline kernel table."""
    gen = torch.Generator().manual_seed(d + 64 * batch + units)
    gb, sw = 64 * 3 * d // 2, 64 * 3 * (d // 128)
    cache = torch.randint(0, 256, (units * gb,), dtype=torch.uint8, generator=gen)
    scales = (torch.rand(units * sw, generator=gen) * 0.015 + 0.005).half()
    x = torch.randn(batch, d, generator=gen).to(torch.bfloat16 if batch > 4 else torch.float16)
    if row is not None:
        x, batch = x[row:row + 1], 1
    slots = torch.randperm(units, generator=gen).numpy()
    rows = np.zeros((units, 5), dtype=np.uint32)
    rows[:, 0] = rows[:, 1] = rows[:, 2] = slots
    rows[:, 3] = np.arange(units)
    for i in bad:
        rows[i, 2] = units + 7   # past the arena: rejected on the device before any access
    core = torch.from_numpy(rows.astype(np.int32)).cuda()
    dev = [t.cuda() for t in (cache, scales, x)]
    y = torch.full((batch, d), float("nan"), dtype=torch.float16, device="cuda")
    y32 = torch.full((batch, d), float("nan"), dtype=torch.float32, device="cuda")
    backend, queue = NativeBackend(table), ReadyQueue(1)
    try:
        backend.bind(d, 64, units, dev[0], dev[1], physical_groups=units, cache_groups=units, queue_capacity=1,
                     batch=batch, y32=y32)
        queue.reset(1)
        queue.seal(0)
        outs = []
        for _ in range(2):   # both ring slots
            backend.enqueue(0, 0, 1, dev[2], y, torch.cuda.current_stream().cuda_stream, core, units, queue,
                            MODE_PROGRESSIVE)
            torch.cuda.synchronize()
            assert backend.complete()
            outs.append(y32.cpu().numpy().copy())
        assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
        assert np.array_equal(y.cpu().numpy().view(np.uint16), outs[0].astype(np.float16).view(np.uint16))
        return outs[0], (rows, cache.numpy(), scales.numpy().view(np.uint16), x), backend.status()
    finally:
        torch.cuda.synchronize()
        backend.close()
        queue.close()


def check(y32, inputs, rows, what):
    _, cache, scales, x = inputs
    d = y32.shape[1]
    for b in sorted({0, len(y32) // 2, len(y32) - 1}):
        xb = x[b].float().half().numpy().view(np.uint16)
        ref = oracle.layer(rows, int(rows[:, 3].max()) + 1, cache, scales, xb, d, 64, threads=8)["y32"].astype(np.float64)
        rel = np.linalg.norm(y32[b] - ref) / np.linalg.norm(ref)
        mx = np.abs(y32[b] - ref).max()
        print(f"{what} row {b}: rel_l2={rel:.3e} max_abs={mx:.3e}", flush=True)
        assert rel <= REL_L2 and mx <= MAX_ABS * max(1.0, np.sqrt(np.mean(ref * ref))), (rel, mx)


@pytest.mark.parametrize("d,batch,units", CASES)
def test_dense_edges(torch_gpu, d, batch, units):
    print(f"case: dense d={d} batch={batch} units={units}", flush=True)
    y32, inputs, status = dense(torch_gpu, d, batch, units)
    assert status == 0, status
    check(y32, inputs, inputs[0], f"d{d} b{batch} u{units}")


@pytest.mark.parametrize("d,batch", [(1024, 7), (4096, 32), (8192, 32)])
def test_dense_bad_descriptor_is_reported_and_left_out(torch_gpu, d, batch):
    print(f"case: dense d={d} batch={batch} with two descriptors past the arena", flush=True)
    y32, inputs, status = dense(torch_gpu, d, batch, 9, bad=(2, 8))
    assert status & STATUS_BAD_DESCRIPTOR, status
    check(y32, inputs, np.delete(inputs[0], (2, 8), axis=0), f"d{d} b{batch} without the rejected units")


def test_dense_launch_writes_no_stamps(torch_gpu):
    """Stamp rows are the waves of a batch-1..4 grid; a dense launch's grids are larger."""
    cfg = config(1024, batch=5, dense=True)
    print(f"case: stamps bound to {cfg.name}", flush=True)
    layer = DeviceLayer(cfg, stamps=True)
    try:
        layer.seal_empty_queue(1)
        layer.run_core(epoch=1)
        sync_and_check_status(torch_gpu, layer)
        assert not layer.stamps.any().item()
    finally:
        layer.close()


@pytest.mark.parametrize("d,batch,units", [(512, 5, 1), (1024, 16, 0), (8192, 32, 9)])
def test_dense_completion_without_the_poll(torch_gpu, d, batch, units):
    """With a bound of zero the reduction's last block does not poll: the word still comes, after the
    outputs, no status bit is raised, and the outputs are those of a launch that polls."""
    torch = torch_gpu
    print(f"case: completion handed over, dense d={d} batch={batch} units={units}", flush=True)
    cfg = config(d, batch=batch, dense=True)
    layer = DeviceLayer(cfg)
    try:
        layer.seal_empty_queue(1)
        layer.k = min(units, layer.k)
        layer.run_core(epoch=1)
        sync_and_check_status(torch, layer)
        want = layer.y32.clone()
        layer.backend.set_spin_limit(0)
        for _ in range(50):   # both ring slots; the poller or a column block ends the launch
            layer.y32.fill_(float("nan"))
            torch.cuda.synchronize()
            layer.run_core(epoch=1)
            deadline = time.monotonic() + 10
            while not layer.backend.complete():
                assert time.monotonic() < deadline
            got = layer.y32.clone()
            sync_and_check_status(torch, layer)
            assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    finally:
        layer.close()


@pytest.mark.parametrize("G,batch", [(128, 1), (8, 1), (16, 3), (128, 2)])
def test_matrix_products_at_other_groups(torch_gpu, G, batch):
    """d = 8192: the plain walk's two-pass down tiles, the packed walk, a pass of fewer than 64 rows
    shared by the batch rows, two passes per batch row."""
    torch = torch_gpu
    cfg = config(8192, G, batch)
    print(f"case: core layer {cfg.name} k={cfg.active}", flush=True)
    layer = DeviceLayer(cfg)
    try:
        layer.seal_empty_queue(1)
        layer.run_core(epoch=1)
        sync_and_check_status(torch, layer)
        check_rows(layer, layer.core_rows[0], cfg.name)
    finally:
        layer.close()


@pytest.mark.parametrize("entry,table", [("fused", None), ("split", [[4]])])
@pytest.mark.parametrize("batch", [2, 3, 4])
def test_batch_rows_have_the_one_row_bits(torch_gpu, batch, entry, table):
    """d = 8192, 64-neuron groups: two and three rows take the kernels of four, and every row gets
    the bits of a launch of its own through either entry point."""
    print(f"case: d=8192 batch={batch} {entry} against one row at a time", flush=True)
    y32, inputs, status = dense(torch_gpu, 8192, batch, 13, table=table)
    assert status == 0, status
    check(y32, inputs, inputs[0], f"d8192 b{batch} {entry}")
    for row in range(batch):
        one, _, status = dense(torch_gpu, 8192, batch, 13, row=row)
        assert status == 0, status
        assert np.array_equal(one[0].view(np.uint32), y32[row].view(np.uint32)), row
