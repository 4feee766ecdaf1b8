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
