"""Arguments of a run through pinned host memory: the caller's arrays against what arrives, at the edges of slices,
pieces and segments (GPU)."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [
    (1,), (3,), (4096,), (4097,),               # below, at and above one slice of 16 KiB
    (262143,), (262147,),                       # around the size from which several threads copy
    (3, 70001, 5),                              # several arguments in one launch
    tuple(range(1, 20)),                        # more arguments than one launch takes
    (1_600_003, 7, 300_001),                    # pieces of 1 MiB that end inside an argument
    (13_000_001,),                              # slices of 512 KiB
])
def test_arguments_arrive(tmp_path, sizes):
    import torch  # noqa: F401
    from fluidml_amd import fluidml, models

    net = models.Net("copies", 1)
    for i, n in enumerate(sizes):
        net.output(net.relu(net.input(f"x{i}", np.float32, (n,))))
    ex = fluidml.Executor.make_plain_greedy("copies")
    ex.compile(net.save(os.path.join(tmp_path, "copies.onnx")))
    rng = np.random.default_rng(5)
    for _ in range(3):  # other values each time: nothing of an earlier run may show
        args = {f"x{i}": rng.standard_normal(n, dtype=np.float32) for i, n in enumerate(sizes)}
        outs = {v.name: np.full(v.shape, -1.0, np.float32) for v in net.outputs}
        assert ex.invoke({**args, **outs}) >= 0
        for i, v in enumerate(net.outputs):
            np.testing.assert_array_equal(outs[v.name], np.maximum(args[f"x{i}"], 0))


@pytest.mark.parametrize("pieces", [0, 1, 64, 65, 1000])  # (64 blocks: from 65 pieces on they take them in turn)
def test_elapsed_belongs_to_the_run_whose_flags_are_up(device, pieces):
    """The time that a transfer_out leaves is there once all flags are, and is that of its own run: runs of nothing
    and of a few milliseconds in turn."""
    import ctypes

    import torch

    from fluidml_amd import cabi

    def alloc(name, size):
        p = ctypes.c_void_p()
        cabi.call(name, size, ctypes.byref(p))
        return p.value

    size, slice_bytes = pieces * 16384, 32768
    slices = max(1, -(-size // slice_bytes))
    src, clock, counters = (alloc("arena_create", max(n, 1)) for n in (size, 8, 4 * (slices + 1)))
    dst, mailbox = (alloc("host_alloc", n) for n in (size, 64 + 4 * slices))
    ctypes.memset(mailbox, 0, 64 + 4 * slices)
    flags = np.ctypeslib.as_array((ctypes.c_uint32 * slices).from_address(mailbox + 64))
    elapsed = ctypes.c_uint64.from_address(mailbox)
    khz = ctypes.c_int()
    cabi.call("clock_khz", ctypes.byref(khz))
    a = torch.randn(4096, 4096, device=device)
    out = torch.empty_like(a)
    torch.mm(a, a, out=out)
    torch.cuda.synchronize()
    stream = torch.cuda.current_stream().cuda_stream
    n = 1 if pieces else 0
    lists = [(ctypes.c_void_p * 1)(dst), (ctypes.c_void_p * 1)(src), (ctypes.c_size_t * 1)(size)]
    print("[case]", pieces, flush=True)
    for turn in range(1, 13):
        begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        cabi.call("transfer_in", 0, None, None, None, clock, stream)
        begin.record()
        for _ in range(8 if turn % 2 else 0):
            torch.mm(a, a, out=out)
        end.record()
        cabi.call("transfer_out", n, *lists, slice_bytes, clock, mailbox, mailbox + 64, counters, turn, stream)
        while not (flags == turn).all():
            if torch.cuda.current_stream().query():
                assert (flags == turn).all(), "the stream is idle but a flag is missing"
        ms = elapsed.value / khz.value
        torch.cuda.synchronize()
        want = begin.elapsed_time(end)
        assert want - 0.05 < ms < want + 0.5, (turn, ms, want)
    for p in (src, clock, counters):
        cabi.call("arena_destroy", p)
    for p in (dst, mailbox):
        cabi.call("host_free", p)


def test_helpers_sleep_while_the_plan_runs(tmp_path):
    """The threads that help with a large output do not poll through the replays in front of it: one thread waits."""
    import time

    import torch  # noqa: F401
    from fluidml_amd import fluidml, models

    net = models.Net("long", 1)
    x = net.input("x", np.float32, (1024, 1024))
    w = net.normal((1024, 1024), std=1 / 32)
    y = x
    for _ in range(8):
        y = net.matmul(y, w)
    net.output(y)  # 4 MiB
    ex = fluidml.Executor.make_plain_greedy("long", 400)
    ex.compile(net.save(os.path.join(tmp_path, "long.onnx")))
    args = {"x": np.ones((1024, 1024), np.float32), net.outputs[0].name: np.zeros((1024, 1024), np.float32)}
    ex.invoke(args)
    wall, cpu = time.perf_counter(), time.process_time()
    ex.invoke(args)
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert wall > 0.02 and cpu < 2.5 * wall, (wall, cpu)  # (the caller and what the runtime itself does; eight with helpers)
