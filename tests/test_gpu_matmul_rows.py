"""Contractions of few rows and short sums (matmul_rows.hip) on the GPU: every tile its rule can pick, at ragged extents, against
a float64 product, and every epilogue against the same call on a tile of matmul.hip that is named."""
import ctypes

import pytest

from test_gpu_matmul_parts import Problem, close
from util import launches

pytestmark = pytest.mark.gpu
STAGED = 1 << 4 | 1 << 8  # FL_TILE_32x32_STAGED, K not split


# the tile by the number of 16x16 tiles, and K: below a stage of 32, between stages, slices without a stage, the longest
@pytest.mark.parametrize("M,K,N", [
    (1, 4, 4), (16, 32, 16), (17, 36, 33), (5, 260, 7), (37, 1152, 49), (77, 2048, 511),  # 16x16
    (100, 36, 600), (129, 772, 516), (128, 1152, 768),                                    # 16x32
    (200, 64, 901), (128, 512, 1536),                                                     # 16x48
    (300, 100, 800), (255, 512, 1003),                                                    # 32x32
    (300, 68, 1150), (256, 544, 1531),                                                    # 32x48
    (140, 40, 4001), (100, 24, 4003), (96, 16, 12547), (33, 4, 20000),                    # waves side by side
])
def test_rows_tiles(device, M, K, N):
    print("[case]", M, K, N, flush=True)
    with Problem(device, M, K, N) as p:
        want = p.x.double() @ p.w[0].double() + p.b[0].double()
        out = p.out()
        assert p.chain(out, 0) == 0
        close(out, want, "rule")
        if K >= 512:
            other = p.out()
            assert p.chain(other, STAGED) == 0
            rel, before = (((t.double() - want).norm() / want.norm()).item() for t in (out, other))
            assert rel <= 1.05 * before  # (eight slices of K where the other tile has four: sums no longer than its)


@pytest.mark.parametrize("M,K,N", [(33, 128, 64), (70, 288, 160), (150, 800, 768), (200, 96, 896), (320, 64, 512), (256, 768, 1440)])
def test_rows_epilogues(device, M, K, N):
    """Bias and chain, addends, siblings with split columns, both forms of a deferred LayerNormalization, row statistics."""
    print("[case]", M, K, N, flush=True)
    with Problem(device, M, K, N, count=2) as p:
        cabi, torch = p.cabi, p.torch
        e1, e2 = p.rand(M, N), p.rand(M, N)
        gamma, beta, c1 = p.rand(N), p.rand(N), [w.sum(0) for w in p.w]
        stats_k, stats_n = (torch.empty(M, w // 32, 2, device=device) for w in (K, N))
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
            none, res = ctypes.byref(cabi.make_chain([])), [p.out()]
            gelu = [(cabi.EW_DIV_C, 2 ** 0.5), (cabi.EW_ERF, 0.0), (cabi.EW_ADD_C, 1.0), (cabi.EW_MUL_X, 0.0), (cabi.EW_MUL_C, 0.5)]
            assert p.chain(res[0], flags, gelu) == 0
            for second in (None, e2):
                out = p.out()
                assert cabi.lib.fluidml_hip_matmul_chain_add(p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), p.ref(out), none, p.ref(e1),
                                                             p.ref(second) if second is not None else None, flags, None) == 0
                res.append(out)
            outs = [torch.full((N // 32, M, 32), 9.0, device=device) for _ in range(2)]  # heads of 32 that a transpose moved apart
            views = [p.tensor(o, (M, N), (32, 1)) for o in outs]
            assert cabi.lib.fluidml_hip_matmul_chain_group(2, p.ref(p.x), p.list(p.w), p.list(p.b), p.list(views), 32,
                                                           cabi.i64_array([32 * M] * 2), none, flags, None) == 0
            res += outs
            outs, n = [p.out() for _ in range(2)], norm(cabi.FL_NORM_LHS, K, stats_k)
            assert cabi.lib.fluidml_hip_matmul_chain_group_norm(2, p.ref(p.x), p.list(p.w), p.list(p.b), p.list(c1), p.list(outs), 0, None, none,
                                                                None, ctypes.byref(n), flags, None) == 0
            res += outs
            deferred = [(cabi.FL_NORM_NONE, 0, None)] + [(cabi.FL_NORM_ADDEND, N, stats_n)] * (N <= 1024)
            for mode, width, given in deferred:
                out, stats = p.out(), torch.full((M, N // 32, 2), 9.0, device=device)
                n = norm(mode, width, given, stats, e2)
                assert cabi.lib.fluidml_hip_matmul_chain_group_norm(1, p.ref(p.x), p.list(p.w[1:]), p.list(p.b[1:]), None, p.list([out]), 0, None,
                                                                    none, p.ref(e1), ctypes.byref(n), flags, None) == 0
                res += [out, stats]
            return res

        for i, (got, want) in enumerate(zip(calls(0), calls(STAGED))):
            close(got, want, f"result {i}")


def test_rows_infinities(device):
    """What lies past M, N and K, repeated to fill a tile, reaches no result."""
    for M, K, N in [(17, 36, 33), (20, 300, 50)]:
        with Problem(device, M, K, N) as p:
            inf = float("inf")
            p.x[M - 1, 0], p.x[3, 0], p.w[0][K - 1, 5], p.w[0][2, N - 1] = inf, float("nan"), -inf, inf
            want = p.x.double() @ p.w[0].double() + p.b[0].double()
            out = p.out()
            assert p.chain(out, 0) == 0
            assert p.torch.equal(out.isnan(), want.isnan()) and p.torch.equal(out.isinf(), want.isinf())
            fine = want.isfinite()
            close(out[fine], want[fine], "finite results")


# 16x16, 32x48, 16x16, 16x128, 16x128, 16x256 (its last workgroup's last waves lie past the pixels), 16x256 (one lane's second column does)
POINTWISE = [(4, 24, 9, 7), (144, 40, 28, 28), (1152, 320, 7, 7), (16, 96, 61, 67), (32, 16, 112, 112), (16, 96, 127, 99), (28, 130, 65, 63)]


@pytest.mark.parametrize("C,F,H,W", POINTWISE)
@pytest.mark.parametrize("in_place", [False, True], ids=["", "in_place"])
def test_rows_pointwise_conv(device, C, F, H, W, in_place):
    """Pointwise convolution with a scale per channel and a skip tensor, both alone and together, odd numbers of pixels; the skip
    tensor may be the result's own memory: every element is read and written by one thread."""
    import torch

    from fluidml_amd import cabi

    print("[case]", C, F, H, W, flush=True)
    g = torch.Generator(device=device)
    g.manual_seed(C + F)
    x, w, b = (torch.randn(*s, device=device, generator=g) for s in ((1, C, H, W), (F, C, 1, 1), (F,)))
    # (weights of C^-1/2 as in Problem: partial sums of size one, rounded C times by 2^-25 each, stay below 1e-5 in the root mean square
    # times four; of unit weights the sums are C^1/2 times larger and where they cancel no relative bound holds)
    w *= C ** -0.5
    scale, skip = torch.randn(1, C, 1, 1, device=device, generator=g), torch.randn(1, F, H, W, device=device, generator=g)
    ref = lambda t: ctypes.byref(cabi.make_tensor(t.data_ptr(), cabi.FL_FLOAT32, t.shape, t.stride()))
    one, relu = cabi.i64_array([1, 1]), cabi.make_chain([(cabi.EW_RELU, 0.0)])
    for s, e in ((scale, None), (None, skip), (scale, skip), (None, None)):
        want = torch.einsum("fc,cp->fp", w.double()[:, :, 0, 0].cpu(), (x * s if s is not None else x).double().cpu().view(C, -1))
        want = (want + b.double().cpu()[:, None]).clamp_min(0).view(1, F, H, W) + (e.double().cpu() if e is not None else 0)
        out = torch.full((1, F, H, W), 9.0, device=device)
        if in_place and e is not None:
            out.copy_(e)
            e = out
        if s is None and e is None:
            cabi.call("conv_chain", ref(x), ref(w), ref(b), ref(out), None, one, one, ctypes.c_int64(1), ctypes.byref(relu), ctypes.c_uint32(0), None)
        else:
            cabi.call("conv_chain_scale_add", ref(x), ref(w), ref(b), ref(out), None, one, one, ctypes.c_int64(1), ctypes.byref(relu),
                      ref(s) if s is not None else None, ref(e) if e is not None else None, ctypes.c_uint32(0), None)
        close(out, want, f"scale {s is not None} skip {e is not None}")


# template arguments: matrix tiles of rows, columns per lane, waves side by side, slices of K
TILES = {"16x16": (1, 1, 1, 8), "16x32": (1, 2, 1, 8), "16x48": (1, 3, 1, 8), "32x32": (2, 2, 1, 8), "32x48": (2, 3, 1, 8),
         "16x128": (1, 2, 4, 2), "16x256": (1, 2, 8, 1)}


def tile_of(call):
    """The tile of the one launch of `call`, None if it is another kernel's."""
    call(None)
    (name, _), = launches(call)
    if "MatmulRowsKernel" not in name:
        return None
    return next(t for t, a in TILES.items() if "MatmulRowsKernelI" + "".join(f"Li{n}E" for n in a) in name)


# both sides of each line the rule draws
@pytest.mark.parametrize("M,K,N,tile", [
    (256, 2048, 256, "16x16"), (256, 2052, 256, None), (257, 1152, 256, "16x32"), (257, 1156, 256, None),
    (192, 320, 768, "16x48"), (192, 384, 768, None), (192, 512, 768, "16x48"), (192, 640, 768, None), (192, 704, 768, "16x48"),
    (192, 128, 768, "16x48"), (192, 896, 768, "16x48"),
    (192, 128, 1024, "32x32"), (192, 384, 1024, None), (192, 640, 1024, None), (192, 896, 1024, "32x32"),
    (512, 128, 768, None), (512, 192, 768, "32x48"), (512, 384, 768, None), (512, 512, 768, "32x48"),
    (128, 384, 768, "16x32"), (128, 640, 768, "16x32"),
    (513, 68, 768, None),
])
def test_rows_rule(device, M, K, N, tile):
    with Problem(device, M, K, N) as p:
        out, none = p.out(), ctypes.byref(p.cabi.make_chain([]))
        assert tile_of(lambda s: p.cabi.call("matmul_chain", p.ref(p.x), p.ref(p.w[0]), p.ref(p.b[0]), p.ref(out), none, 0, s)) == tile


@pytest.mark.parametrize("C,F,pixels,tile,scaled", [
    (64, 256, 6144, "16x128", "16x128"),   # 768 workgroups
    (64, 256, 6272, None, None),           # 784
    (48, 128, 12544, None, None),
    (64, 96, 12544, "16x128", "16x128"),   # 64 rows pad a third
    (64, 112, 25600, None, None),          # and less
    (40, 1024, 6400, None, None),
    (24, 256, 4096, "16x256", "16x256"),   # 256 workgroups
    (24, 256, 4224, "16x256", None),
    (32, 1024, 6400, "16x256", None),
    (16, 112, 25600, "16x256", "16x256"),  # 64 rows pad a seventh
    (16, 120, 25600, "16x256", None),
])
def test_rows_rule_pointwise(device, C, F, pixels, tile, scaled):
    import torch

    from fluidml_amd import cabi

    x, w, b = (torch.zeros(*s, device=device) for s in ((1, C, pixels, 1), (F, C, 1, 1), (F,)))
    scale, out = torch.zeros(1, C, 1, 1, device=device), torch.zeros(1, F, pixels, 1, device=device)
    ref = lambda t: ctypes.byref(cabi.make_tensor(t.data_ptr(), cabi.FL_FLOAT32, t.shape, t.stride()))
    one, none = cabi.i64_array([1, 1]), ctypes.byref(cabi.make_chain([]))
    assert tile_of(lambda s: cabi.call("conv_chain", ref(x), ref(w), ref(b), ref(out), None, one, one, ctypes.c_int64(1), none,
                                       ctypes.c_uint32(0), s)) == tile
    assert tile_of(lambda s: cabi.call("conv_chain_scale_add", ref(x), ref(w), ref(b), ref(out), None, one, one, ctypes.c_int64(1), none,
                                       ref(scale), None, ctypes.c_uint32(0), s)) == scaled
