"""Contractions against packed weights (fluidml_hip_contract_pack) on the GPU: every tile at its edges, with K split over
workgroups, against a float64 product; every epilogue against the same call before the weights were packed; and the
values its bf16 parts cannot carry."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TILES = {"32x64": 9, "64x64": 10, "64x128": 11, "64x128_K2": 12}
UNSUPPORTED = -8


class Problem:
    """x [M, K] against `count` weights [K, N] (or [N, K]), their packed forms held while the object lives."""

    def __init__(self, device, M, K, N, count=1, trans_b=False, seed=0, scale=1.0):
        import torch

        from fluidml_amd import cabi

        self.torch, self.cabi, self.M, self.K, self.N = torch, cabi, M, K, N
        g = torch.Generator(device=device)
        g.manual_seed(seed + M * 7 + K * 3 + N)
        self.rand = lambda *s: torch.randn(*s, device=device, generator=g)
        self.x = self.rand(M, K) * scale
        self.w = [self.rand(*((N, K) if trans_b else (K, N))) * K ** -0.5 for _ in range(count)]
        self.b = [self.rand(N) for _ in range(count)]
        self.trans_b, self.packed = trans_b, []

    def pack(self, parts=3):
        for w in self.w:
            p, n = ctypes.c_void_p(), ctypes.c_size_t()
            # (a number of rows at which packing is always worth it: the small problems here test the edges)
            self.cabi.call("contract_pack", self.ref(w), int(self.trans_b), 1 << 40, parts, None, ctypes.byref(p), ctypes.byref(n))
            self.packed.append(p)

    def __enter__(self):
        return self

    def __exit__(self, *_):
        self.torch.cuda.synchronize()
        for p in self.packed:
            self.cabi.call("contract_unpack", p)

    def tensor(self, t, shape=None, strides=None):
        return self.cabi.make_tensor(t.data_ptr(), self.cabi.FL_FLOAT32, shape or t.shape, strides or t.stride())

    def ref(self, t, shape=None, strides=None):
        return ctypes.byref(self.tensor(t, shape, strides))

    def list(self, ts):
        ptr = ctypes.POINTER(self.cabi.FlTensor)
        return (ptr * len(ts))(*[ctypes.pointer(t if isinstance(t, self.cabi.FlTensor) else self.tensor(t)) for t in ts])

    def out(self):
        return self.torch.full((self.M, self.N), 9.0, device=self.x.device)

    def chain(self, out, flags, steps=()):
        return self.cabi.lib.fluidml_hip_matmul_chain(self.ref(self.x), self.ref(self.w[0]), self.ref(self.b[0]), self.ref(out),
                                                      ctypes.byref(self.cabi.make_chain(steps)), flags, None)


def flags_of(tile, splits=1):
    return TILES[tile] << 4 | splits << 8


def close(got, want, what):
    got, want = got.double().cpu().numpy(), want.double().cpu().numpy()
    assert np.isfinite(got).all(), what
    err = np.abs(got - want)
    assert (err <= 1e-5 + 1e-4 * np.abs(want)).all(), f"{what}: max err {err.max():.3e}"


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,K,N", [
    (1, 8, 1), (32, 16, 32), (33, 24, 65), (63, 128, 127), (65, 136, 129), (127, 248, 33), (128, 256, 128), (129, 520, 257), (40, 768, 64),
])
def test_packed_tiles(device, tile, M, K, N):
    print("[case]", tile, M, K, N, flush=True)
    with Problem(device, M, K, N) as p:
        want = p.x.double() @ p.w[0].double() + p.b[0].double()
        p.pack()
        ran = 0
        for splits in (1, 2, 3, 8):
            for _ in range(2):  # (again: the arrival counters are back at zero)
                out = p.out()
                rc = p.chain(out, flags_of(tile, splits))
                if rc == UNSUPPORTED:
                    assert splits > 1  # too few chunks of K
                    continue
                assert rc == 0
                close(out, want, f"{tile} {splits} splits")
                ran += 1
        assert ran >= 2
        if K >= 512:
            rel = ((out.double() - want).norm() / want.norm()).item() if rc == 0 else 0.0
            assert rel < 1.5e-7  # (the fp32 instruction: 1.8e-7 at 768 products)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,pad", [(64, 64, 0), (66, 72, 1), (97, 130, 3), (131, 33, 0)])
def test_packed_results_with_rows_side_by_side(device, tile, M, N, pad):
    """The result's rows at unit stride, runs of four of them whole and cut off, at addresses that are no multiple of 16 bytes."""
    with Problem(device, M, 256, N) as p:
        p.pack()
        out = p.torch.full((N * (M + pad) + 4,), 9.0, device=device)
        for first in (0, 1):
            view = out[first:]
            ref = p.ref(view, (M, N), (1, M + pad))
            rc = p.cabi.lib.fluidml_hip_matmul_chain(p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), ref, ctypes.byref(p.cabi.make_chain([])),
                                                     flags_of(tile), None)
            assert rc == 0
            got = p.torch.as_strided(view, (M, N), (1, M + pad))
            close(got, p.x.double() @ p.w[0].double() + p.b[0].double(), "transposed")
            if pad:
                assert (p.torch.as_strided(view, (N - 1, pad), (M + pad, 1), view.storage_offset() + M) == 9.0).all()
            out.fill_(9.0)


@pytest.mark.parametrize("tile", TILES)
def test_packed_bf16(device, tile):
    for M, K, N in [(33, 264, 65), (128, 768, 96)]:
        with Problem(device, M, K, N) as p:
            want = p.x.bfloat16().double() @ p.w[0].bfloat16().double() + p.b[0].double()
            p.pack(1)
            out = p.out()
            assert p.chain(out, flags_of(tile) | p.cabi.FL_CONTRACT_BF16) == 0
            close(out, want, "bf16")
            assert p.chain(out, flags_of(tile)) == UNSUPPORTED  # (packed for the other precision)


@pytest.mark.parametrize("tile,splits", [(t, s) for t in TILES for s in (1, 2)])
def test_packed_epilogues(device, tile, splits):
    """Bias and elementwise chain, addends, siblings with split columns, both forms of a deferred LayerNormalization,
    row statistics: each call before packing (any tile) and after (this tile)."""
    M, K, N = 70, 288, 160
    print("[case]", tile, splits, flush=True)
    with Problem(device, M, K, N, count=3) as p:
        cabi, torch = p.cabi, p.torch
        e1, e2, x3 = p.rand(M, N), p.rand(M, N), p.rand(M, K)
        gamma, beta, c1 = p.rand(N), p.rand(N), [w.sum(0) for w in p.w]
        stats_k = torch.empty(M, K // 32, 2, device=device)
        stats_n = torch.empty(M, N // 32, 2, device=device)
        for stats, t in ((stats_k, p.x), (stats_n, e1)):
            runs = t.reshape(M, -1, 32)
            stats[..., 0] = runs.mean(-1)
            stats[..., 1] = ((runs - runs.mean(-1, keepdim=True)) ** 2).sum(-1)

        def norm(deferred, width=0, stats=None, stats_out=None, addend2=None):
            n = cabi.FlNormFusion()
            n.deferred, n.width, n.epsilon = deferred, width, 1e-5
            n.stats = stats.data_ptr() if stats is not None else None
            n.stats_out = stats_out.data_ptr() if stats_out is not None else None
            if deferred == cabi.FL_NORM_ADDEND:
                n.scale, n.shift = ctypes.pointer(p.tensor(gamma)), ctypes.pointer(p.tensor(beta))
            if addend2 is not None:
                n.addend2 = ctypes.pointer(p.tensor(addend2))
            return n

        def calls(flags):
            res = []
            out = p.out()
            gelu = [(cabi.EW_DIV_C, 2 ** 0.5), (cabi.EW_ERF, 0.0), (cabi.EW_ADD_C, 1.0), (cabi.EW_MUL_X, 0.0), (cabi.EW_MUL_C, 0.5)]
            assert p.chain(out, flags, gelu) == 0
            res.append(out)
            out = p.out()
            none = ctypes.byref(cabi.make_chain([]))
            assert cabi.lib.fluidml_hip_matmul_chain_add(p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), p.ref(out), none, p.ref(e1), p.ref(e2), flags, None) == 0
            res.append(out)
            # siblings, 160 columns as 5 heads of 32 that a transpose moved apart: [5, M, 32]
            outs = [torch.full((5, M, 32), 9.0, device=device) for _ in range(3)]
            views = [p.tensor(o, (M, N), (32, 1)) for o in outs]
            outer = cabi.i64_array([32 * M] * 3)
            assert cabi.lib.fluidml_hip_matmul_chain_group(3, p.ref(p.x), p.list(p.w), p.list(p.b), p.list(views), 32, outer, none, flags, None) == 0
            res += outs
            # LayerNormalization of the left operand, two projections
            outs = [p.out() for _ in range(2)]
            n = norm(cabi.FL_NORM_LHS, K, stats_k)
            assert cabi.lib.fluidml_hip_matmul_chain_group_norm(2, p.ref(p.x), p.list(p.w[:2]), p.list(p.b[:2]), p.list(c1[:2]), p.list(outs), 0, None, none,
                                                                None, ctypes.byref(n), flags, None) == 0
            res += outs
            # LayerNormalization of the addend, a second addend, statistics of the result
            out, stats = p.out(), torch.full((M, N // 32, 2), 9.0, device=device)
            n = norm(cabi.FL_NORM_ADDEND, N, stats_n, stats, e2)
            assert cabi.lib.fluidml_hip_matmul_chain_group_norm(1, p.ref(x3), p.list(p.w[2:]), p.list(p.b[2:]), None, p.list([out]), 0, None, none,
                                                                p.ref(e1), ctypes.byref(n), flags, None) == 0
            return res + [out, stats]

        want = calls(0)
        p.pack()
        for i, (got, ref) in enumerate(zip(calls(flags_of(tile, splits)), want)):
            close(got, ref, f"result {i}")


def test_packed_addend_keeps_four_to_a_unit(device):
    """bf16 launches of 64x128 tiles with an addend hold no registers for the second one that none of them has."""
    from util import launched

    with Problem(device, 128, 256, 33000) as p:
        e = p.rand(128, 33000)
        p.pack(1)
        out = p.out()
        none = ctypes.byref(p.cabi.make_chain([]))
        call = lambda s: p.cabi.call("matmul_chain_add", p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), p.ref(out), none, p.ref(e), None,
                                     p.cabi.FL_CONTRACT_BF16, s)
        (name, fit, _, scratch), = launched(call, first_on_its_stream=True)
        assert "MatmulPartsKernelILi1ELi2ELi4ELi1E" in name and fit >= 4 and scratch == 0, (name, fit, scratch)
        close(out, p.x.bfloat16().double() @ p.w[0].bfloat16().double() + p.b[0].double() + e.double(), "addend")


def test_packed_gemm(device):
    with Problem(device, 48, 200, 72, trans_b=True) as p:
        def call(flags):
            out = p.out()
            none = ctypes.byref(p.cabi.make_chain([]))
            assert p.cabi.lib.fluidml_hip_gemm_chain(p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), p.ref(out), 0.5, 2.0, 0, 1, none, flags, None) == 0
            return out
        want = call(0)
        p.pack()
        close(call(flags_of("32x64")), want, "gemm")


@pytest.mark.parametrize("tile", TILES)
def test_packed_outside_the_parts(device, tile):
    """Infinities and NaN behave as in fp32, and operands whose parts would be denormal keep their precision."""
    with Problem(device, 70, 200, 100) as p:
        p.x[3, 7], p.x[69, 199], p.w[0][11, 99] = float("inf"), float("nan"), float("-inf")
        want = p.x.double() @ p.w[0].double() + p.b[0].double()
        p.pack()
        out = p.out()
        assert p.chain(out, flags_of(tile)) == 0
        assert p.torch.equal(out.isnan(), want.isnan()) and p.torch.equal(out.isinf(), want.isinf())
        fine = want.isfinite()
        close(out[fine], want[fine], "finite results beside infinities")
    with Problem(device, 40, 96, 64, scale=1e-36) as p:
        p.x.abs_()
        p.w[0].abs_()
        p.b[0].zero_()
        want = p.x.double() @ p.w[0].double()
        p.pack()
        out = p.out()
        assert p.chain(out, flags_of(tile)) == 0
        np.testing.assert_allclose(out.double().cpu().numpy(), want.cpu().numpy(), rtol=1e-5)


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("x_scale,w_scale", [(1e-42, 1.0), (1e-41, 1e-3), (1e-21, 2e-18), (1e-26, 1e-16)])
def test_packed_products_that_vanish(device, tile, x_scale, w_scale):
    """Results of denormal numbers: where parts or their products come to nothing, the fp32 instruction has the word.
    Its sums round to multiples of 2^-149, half of one per product; without the second pass they were all zero."""
    M, K, N = 40, 96, 64
    with Problem(device, M, K, N) as p:
        # (no exact zeros, weights from 2^-60 on)
        p.x.copy_((p.x.abs() + 0.5).double() * x_scale)
        p.w[0].copy_((p.w[0].abs() + 0.5) * w_scale)
        p.x[3] = 0
        p.x[5, :7] = 0
        p.x[7, 1:] = 0
        p.b[0].zero_()
        want = p.x.double() @ p.w[0].double()
        p.pack()
        out = p.out()
        assert p.chain(out, flags_of(tile)) == 0
        err = (out.double() - want).abs()
        assert (err <= K * 2.0 ** -150 + 1e-6 * want.abs()).all(), err.max().item()
        assert (out[3] == 0).all() and (out[7] != 0).any()


@pytest.mark.parametrize("element,value", [(0, 2.0 ** -61), (95 * 64 + 63, -1e-40), (77, 2.0 ** 20), (6143, -3e38)])
def test_weights_the_parts_cannot_carry_are_not_packed(device, element, value):
    """Refused, and the contraction runs on them as they stand; zeros, infinities and NaN are no reason."""
    with Problem(device, 40, 96, 64, scale=1e-35) as p:
        p.w[0].view(-1)[5] = 0.0
        keep = p.w[0].view(-1)[element].item()
        p.w[0].view(-1)[element] = value
        want = p.x.double() @ p.w[0].double() + p.b[0].double()
        with pytest.raises(p.cabi.FluidmlHipError) as e:
            p.pack()
        assert e.value.code == UNSUPPORTED
        out = p.out()
        assert p.chain(out, flags_of("32x64")) == UNSUPPORTED and p.chain(out, 0) == 0
        close(out, want, "as they stand")
        p.w[0].view(-1)[element] = keep
        p.w[0].view(-1)[6], p.w[0].view(-1)[7] = float("inf"), float("nan")
        p.pack()


@pytest.mark.parametrize("M,K,N", [  # 64x128 tiles times splits of the rule
    (77, 768, 16512),                   # more than 256
    (256, 640, 8192), (192, 768, 5504),  # 256, 129
    (256, 1280, 4096), (256, 1272, 4096),  # 128 x 2, the next shorter K
    (150, 1920, 4000), (140, 2560, 2048), (68, 2560, 4224),  # 96 x 2, 48 x 4, 66 x 3
    (96, 1288, 2060),                   # not packed in three parts
])
def test_packed_tiles_of_the_rule(device, M, K, N):
    for parts in (3, 1):
        with Problem(device, M, K, N) as p:
            x, w = (p.x, p.w[0]) if parts == 3 else (p.x.bfloat16(), p.w[0].bfloat16())
            want = x.double() @ w.double() + p.b[0].double()
            p.pack(parts)
            got = ctypes.c_int32()
            p.cabi.call("take_packed_parts", ctypes.byref(got))
            print("[case]", M, K, N, parts, flush=True)
            for _ in range(2):
                out = p.out()
                assert p.chain(out, 0 if parts == 3 else p.cabi.FL_CONTRACT_BF16) == 0
                close(out, want, f"{parts} parts")
            p.cabi.call("take_packed_parts", ctypes.byref(got))
            assert got.value == (parts if parts == 1 or (M * N >= 280000 and float(M) * K * N >= 5.8e8) else 0)


@pytest.mark.parametrize("M", [65, 77, 95, 96, 97])  # tiles of 96 rows, their last rows missing or all there, and one row more
@pytest.mark.parametrize("K,N", [(712, 32800), (1160, 32769)])  # 257 of 128 columns, the last chunk of K a quarter full
def test_packed_tiles_of_96_rows(device, M, K, N):
    with Problem(device, M, K, N) as p:
        p.pack()
        out = p.out()
        print("[case]", M, K, N, flush=True)
        assert p.chain(out, 0, [(p.cabi.EW_RELU, 0.0)]) == 0
        close(out, (p.x.double() @ p.w[0].double() + p.b[0].double()).clamp(min=0), "rows")


def _ran_on_96_rows(call, extra):
    from util import launched

    (name, fit, _, scratch), = launched(call, first_on_its_stream=True)
    assert "MatmulPartsKernelILi3ELi3ELi4ELi1E" in name and f"ELi{extra}EEE" in name and fit >= 2 and scratch == 0, (name, fit, scratch)


@pytest.mark.parametrize("M", [65, 77, 96])
def test_packed_epilogues_of_96_rows(device, M):
    """Each epilogue that a launch of the rule's tile of 96 rows can have, before packing (any tile) and after."""
    K = 296  # the last chunk a quarter full

    def norm(cabi, stats=None, out=None):
        n = cabi.FlNormFusion()
        n.deferred, n.width, n.epsilon = (cabi.FL_NORM_LHS, K, 1e-5) if stats is not None else (cabi.FL_NORM_NONE, 0, 0.0)
        n.stats = stats.data_ptr() if stats is not None else None
        n.stats_out = out.data_ptr() if out is not None else None
        return n

    def row_stats(torch, t):
        runs = t.split(32, -1)
        return torch.stack([torch.stack([r.mean(-1), ((r - r.mean(-1, keepdim=True)) ** 2).sum(-1)], -1) for r in runs], 1).contiguous()

    # 257 tiles of one contraction; 86 of each of three members
    for N, count in ((32800, 1), (11008, 3)):
        print("[case]", M, K, N, count, flush=True)
        with Problem(device, M, K, N, count=count) as p:
            cabi, torch = p.cabi, p.torch
            none = ctypes.byref(cabi.make_chain([]))
            relu = ctypes.byref(cabi.make_chain([(cabi.EW_RELU, 0.0)]))
            stats, c1 = row_stats(torch, p.x), [w.sum(0) for w in p.w]
            e1, e2 = p.rand(M, N), p.rand(M, N)

            def cases():
                if count == 1:
                    out = p.out()
                    yield 1, [out], lambda s: cabi.call("matmul_chain_add", p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), p.ref(out), relu, p.ref(e1), None, 0, s)
                    out2 = p.out()
                    yield 1, [out2], lambda s: cabi.call("matmul_chain_add", p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), p.ref(out2), none, p.ref(e1), p.ref(e2), 0, s)
                    out3, stats_n = p.out(), torch.full((M, 1025, 2), 9.0, device=device)
                    n3 = norm(cabi, out=stats_n)
                    yield 1, [out3, stats_n], lambda s: cabi.call("matmul_chain_group_norm", 1, p.ref(p.x), p.list(p.w), p.list(p.b), None, p.list([out3]), 0, None,
                                                                  none, p.ref(e1), ctypes.byref(n3), 0, s)
                    out4 = torch.full((N, M + 1), 9.0, device=device)
                    yield 0, [out4], lambda s: cabi.call("matmul_chain", p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), p.ref(out4, (M, N), (1, M + 1)), none, 0, s)
                outs = [p.out() for _ in range(count)]
                n5 = norm(cabi, stats=stats)
                yield 1, outs, lambda s: cabi.call("matmul_chain_group_norm", count, p.ref(p.x), p.list(p.w), p.list(p.b), p.list(c1), p.list(outs), 0, None,
                                                   none, None, ctypes.byref(n5), 0, s)
                if count > 1:  # columns as heads of 32 that a transpose moved apart
                    heads = [torch.full((N // 32, M, 32), 9.0, device=device) for _ in range(count)]
                    views = [p.tensor(o, (M, N), (32, 1)) for o in heads]
                    outer = cabi.i64_array([32 * M] * count)
                    yield 0, heads, lambda s: cabi.call("matmul_chain_group", count, p.ref(p.x), p.list(p.w), p.list(p.b), p.list(views), 32, outer, none, 0, s)

            want = []
            for _, outs, call in cases():
                call(None)
                want.append([o.clone() for o in outs])
            p.pack()
            for i, (extra, outs, call) in enumerate(cases()):
                _ran_on_96_rows(call, extra)
                for got, ref in zip(outs, want[i]):
                    close(got, ref, f"case {i}")


@pytest.mark.parametrize("M", [65, 96])
def test_packed_96_rows_outside_the_parts(device, M):
    K, N = 296, 32800
    with Problem(device, M, K, N) as p:
        p.x[3, 7], p.x[M - 1, K - 1], p.w[0][11, N - 1] = float("inf"), float("nan"), float("-inf")
        want = p.x.double() @ p.w[0].double() + p.b[0].double()
        p.pack()
        out = p.out()
        _ran_on_96_rows(lambda s: p.cabi.call("matmul_chain", p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), p.ref(out), ctypes.byref(p.cabi.make_chain([])), 0, s), 0)
        assert p.torch.equal(out.isnan(), want.isnan()) and p.torch.equal(out.isinf(), want.isinf())
        fine = want.isfinite()
        close(out[fine], want[fine], "finite results beside infinities")
    for x_scale, w_scale in ((1e-41, 1e-3), (1e-21, 2e-18)):  # products that vanish (weights from 2^-60 on)
        with Problem(device, M, K, N) as p:
            p.x.copy_((p.x.abs() + 0.5).double() * x_scale)
            p.w[0].copy_((p.w[0].abs() + 0.5) * w_scale)
            p.x[3] = 0
            p.x[5, :7] = 0
            p.x[7, 1:] = 0
            p.b[0].zero_()
            want = p.x.double() @ p.w[0].double()
            p.pack()
            out = p.out()
            _ran_on_96_rows(lambda s: p.cabi.call("matmul_chain", p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), p.ref(out), ctypes.byref(p.cabi.make_chain([])), 0, s), 0)
            err = (out.double() - want).abs()
            assert (err <= K * 2.0 ** -150 + 1e-6 * want.abs()).all(), err.max().item()
            assert (out[3] == 0).all() and (out[7] != 0).any()


def test_a_plan_frees_the_packed_weights_no_launch_takes(device, tmp_path, monkeypatch):
    """The tile configuration of a contraction is picked after its weights have been packed."""
    import json
    import os

    from fluidml_amd import fluidml, models

    net = models.Net("two", 1)
    x = net.input("x", np.float32, (512, 768))
    net.output(net.add(net.matmul(x, net.normal((768, 3072))), net.zeros((3072,))))
    net.output(net.matmul(net.relu(x), net.normal((768, 2560))))
    path = net.save(os.path.join(tmp_path, "two.onnx"))
    feed = {"x": np.random.default_rng(2).standard_normal((512, 768), np.float32)}
    want = [feed["x"] @ net.initializers[0].const, np.maximum(feed["x"], 0) @ net.initializers[2].const]

    def compiled(tune, packed="1"):
        monkeypatch.setenv("FLUIDML_TUNE", tune)
        monkeypatch.setenv("FLUIDML_MATMUL_PACKED", packed)
        ex = fluidml.Executor.make_plain_greedy("two")
        ex.compile(path)
        outs = {v.name: np.zeros(v.shape, np.float32) for v in net.outputs}
        ex.invoke({**feed, **outs})
        for v, w in zip(net.outputs, want):
            np.testing.assert_allclose(outs[v.name], w, rtol=1e-4, atol=1e-5)
        plan = ex.plan()
        assert plan["peak_device_bytes"] == plan["arena_bytes"] + plan["constant_bytes"] + plan["interface_bytes"] + plan["private_bytes"]
        return ex, plan["private_bytes"], plan["constant_bytes"]

    _, none, full = compiled("0", "0")
    ex, both, rest = compiled("0")
    assert both - none == 768 * (3072 + 2560) * 6 and full - rest == 768 * (3072 + 2560) * 4
    signature = next(sig for sig, _, _ in ex.contraction_choices() if "3072" in sig)
    table = os.path.join(tmp_path, "picks.json")
    with open(table, "w") as f:
        json.dump({signature: {"tile": 2, "splits": 0}}, f)
    _, one, rest = compiled(table)
    assert one - none == 768 * 2560 * 6 and full - rest == 768 * 2560 * 4


@pytest.mark.parametrize("graph", ["1", "0"])
def test_weights_that_exist_packed_only(device, tmp_path, monkeypatch, graph):
    """A plan keeps the one form of its weights that its launches read, both where somebody reads them as they stand; the
    second pass of what the parts cannot carry works from either."""
    import os

    from fluidml_amd import fluidml, models

    monkeypatch.setenv("FLUIDML_TUNE", "0")
    monkeypatch.setenv("FLUIDML_HIP_GRAPH", graph)
    net = models.Net("forms", 1)
    x = net.input("x", np.float32, (512, 768))
    y = net.input("y", np.float32, (768, 2560))
    few = net.input("few", np.float32, (9, 768))
    w = [net.normal((768, n)) for n in (3072, 2560, 2816)]
    net.output(net.matmul(x, w[0]))                    # packed only
    net.output(net.matmul(net.relu(x), w[1]))
    net.output(net.add(y, w[1]))                       # as they stand too
    net.output(net.relu(net.matmul(x, w[2])))
    net.output(net.matmul(few, w[2]))                  # too few rows for the packed form
    conv = net.normal((64, 32, 3, 3), std=0.06)
    img = net.input("img", np.float32, (1, 32, 30, 30))
    net.output(net.relu(net.conv(img, conv, None, [1, 1], [1, 1, 1, 1])))
    ex = fluidml.Executor.make_plain_greedy("forms")
    ex.compile(net.save(os.path.join(tmp_path, "forms.onnx")))
    plan = ex.plan()
    assert plan["constant_bytes"] == 768 * (2560 + 2816) * 4
    assert plan["private_bytes"] >= 768 * (3072 + 2560 + 2816) * 6 + 64 * 32 * 9 * 6
    rng = np.random.default_rng(2)
    for turn in range(3):
        feed = {v.name: rng.standard_normal(v.shape, np.float32) for v in net.inputs}
        if turn == 1:
            feed["x"] *= np.float32(1e-37)
            feed["img"][:] *= np.float32(1e-37)
        if turn == 2:
            feed["x"][5, 7], feed["img"][0, 3, 3, 3] = np.inf, np.nan
        outs = {v.name: np.full(v.shape, 9.0, np.float32) for v in net.outputs}
        ex.invoke({**feed, **outs})
        f64 = {k: v.astype(np.float64) for k, v in feed.items()}
        c = [v.const.astype(np.float64) for v in w]
        with np.errstate(invalid="ignore"):
            pad = np.pad(f64["img"][0], ((0, 0), (1, 1), (1, 1)))
            image = sum(np.tensordot(conv.const[:, :, i, j].astype(np.float64), pad[:, i:i + 30, j:j + 30], 1) for i in range(3) for j in range(3))
            want = [f64["x"] @ c[0], np.maximum(f64["x"], 0) @ c[1], f64["y"] + c[1], np.maximum(f64["x"] @ c[2], 0), f64["few"] @ c[2],
                    np.maximum(image, 0)[None]]
        scale = 1e-37 if turn == 1 else 1.0
        for i, (v, ref) in enumerate(zip(net.outputs, want)):
            got, s = outs[v.name], scale if i in (0, 1, 3, 5) else 1.0
            assert np.array_equal(np.isfinite(got), np.isfinite(ref)), (turn, i)
            fine = np.isfinite(ref)
            assert (np.abs(got[fine] - ref[fine]) <= 1e-5 * s + 1e-5 * np.abs(ref[fine])).all(), (turn, i)


@pytest.mark.parametrize("tile", TILES)
def test_adopted_weights(device, tile):
    """The packed form stands for the weights; calls that would read them as they stood are refused."""
    for trans_b in (False, True):
        with Problem(device, 70, 200, 100, trans_b=trans_b) as p:
            cabi = p.cabi
            w = p.w[0].t() if trans_b else p.w[0]
            p.x[3, 7], p.x[69, 199] = float("inf"), float("nan")
            w[11, 99] = float("-inf")
            want = p.x.double() @ w.double()
            tiny = p.x.clone().nan_to_num_(0, 0, 0).abs_() * 1e-36
            want_tiny = tiny.double() @ w.double()
            p.pack()
            cabi.call("contract_adopt", p.packed[0])
            rhs = cabi.make_tensor(p.packed[0].value, cabi.FL_FLOAT32, p.w[0].shape, p.w[0].stride())
            p.w[0].fill_(float("nan"))
            none, zero = ctypes.byref(cabi.make_chain([])), p.torch.zeros(100, device=device)

            def call(x, flags, rows=70):
                out = p.out()
                rc = cabi.lib.fluidml_hip_gemm_chain(p.ref(x, (rows, 200)), ctypes.byref(rhs), p.ref(zero), p.ref(out, (rows, 100)), 1.0, 1.0, 0,
                                                     int(trans_b), none, flags, None)
                return rc, out

            rc, out = call(p.x, flags_of(tile))
            assert rc == 0 and p.torch.equal(out.isnan(), want.isnan()) and p.torch.equal(out.isinf(), want.isinf())
            fine = want.isfinite()
            close(out[fine], want[fine], "finite results beside infinities")
            rc, out = call(tiny, flags_of(tile))
            fine = want_tiny.isfinite()
            assert rc == 0 and not out[~fine].isfinite().any()
            # (the weights' signs differ: against sums of magnitudes, about 200 times 0.8 times 0.06)
            assert ((out[fine].double() - want_tiny[fine]).abs() <= 1e-6 * 10 * 1e-36).all()
            for flags, rows in ((0, 70), (0, 3), (1 << 4, 70), (3 << 4, 70), (cabi.FL_CONTRACT_BF16, 70)):
                assert call(p.x, flags, rows)[0] == UNSUPPORTED


@pytest.mark.parametrize("M,K,N,count,packed", [
    (65, 768, 11648, 1, True), (64, 768, 12288, 1, False),                                # rows
    (384, 3072, 768, 1, True), (364, 3072, 768, 1, False),                                # results
    (246, 768, 3072, 1, True), (245, 768, 3072, 1, False), (328, 768, 768, 3, True), (327, 768, 768, 3, False),  # products
])
def test_the_rule_counts_rows_results_and_products_of_all_members(device, M, K, N, count, packed):
    with Problem(device, M, K, N, count=count) as p:
        p.pack()
        parts = ctypes.c_int32()
        p.cabi.call("take_packed_parts", ctypes.byref(parts))
        outs = [p.out() for _ in range(count)]
        none = ctypes.byref(p.cabi.make_chain([]))
        assert p.cabi.lib.fluidml_hip_matmul_chain_group(count, p.ref(p.x), p.list(p.w), p.list(p.b), p.list(outs), 0, None, none, 0, None) == 0
        p.cabi.call("take_packed_parts", ctypes.byref(parts))
        assert (parts.value == 3) == packed
        for o, w, b in zip(outs, p.w, p.b):
            close(o, p.x.double() @ w.double() + b.double(), "members")
