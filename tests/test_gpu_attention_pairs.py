"""Attention where a workgroup takes two tiles of queries (more than 256 keys, more than 256 tiles), and the forms its operands
come in (no mask, mask, condition, both; head columns at no unit stride; more batch dims than two; divisors that are powers of
two and others), against float64."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def ref(t):
    import torch

    from fluidml_amd import cabi

    kind = cabi.FL_BOOL if t.dtype == torch.bool else cabi.FL_FLOAT32
    return ctypes.byref(cabi.make_tensor(t.data_ptr(), kind, t.shape, t.stride()))


def run(device, batch, sq, skv, d, masked, where, turned, divisor, spoil=False):
    import torch

    from fluidml_amd import cabi

    print("[case]", batch, sq, skv, d, masked, where, turned, divisor, flush=True)
    g = torch.Generator(device=device)
    g.manual_seed(sq + skv + d)

    def draw(*shape):
        """uniform in -1 .. 1; `turned`: the batch dims lie in the other order, the last two transposed"""
        if not turned:
            return torch.rand(*shape, device=device, generator=g) * 2 - 1
        t = torch.rand(*shape[:-2][::-1], shape[-1], shape[-2], device=device, generator=g) * 2 - 1
        n = len(shape) - 2
        return t.permute(*range(n - 1, -1, -1), n + 1, n)

    q, kt, v = draw(*batch, sq, d), draw(*batch, d, skv), draw(*batch, skv, d)
    mask = torch.rand(*[1] * len(batch), 1, skv, device=device, generator=g) * -8 if masked else None
    cond = torch.ones(sq, skv, dtype=torch.bool, device=device).tril(skv - sq).view(*[1] * len(batch), sq, skv) if where else None
    if spoil:
        q[..., 21, 3] = float("nan")        # second tile of a workgroup
        mask[..., skv - 60:] = -float("inf")  # the last wave has no key left
        v[..., 0, 5] = float("inf")
    fill = float(torch.finfo(torch.float32).min)
    out = torch.full((*batch, sq, d), 9.0, device=device)
    cabi.call("attention", ref(q), ref(kt), ref(v), ref(out), ctypes.c_double(divisor), 1, ref(mask) if masked else None,
              ref(cond) if where else None, ctypes.c_double(fill), None)
    s = torch.matmul(q.double().cpu(), kt.double().cpu()) / divisor
    if masked:
        s = s + mask.double().cpu()
    if where:
        s = torch.where(cond.cpu(), s, torch.tensor(fill, dtype=torch.float64))
    return out.double().cpu(), torch.matmul(torch.softmax(s, -1), v.double().cpu())


@pytest.mark.parametrize("batch,sq,skv,d,turned,divisor", [
    ((17,), 256, 512, 64, False, 8.0),       # whole tiles
    ((9,), 465, 389, 64, False, 7.0),        # one query in the last workgroup (of its first tile); ragged keys
    ((20,), 213, 257, 16, False, 0.5),       # 21 queries there
    ((2, 3, 3), 257, 300, 32, False, 5.0),   # one query
    ((2, 3, 3), 250, 300, 64, True, 8.0),    # three batch dims that do not merge; no unit strides: one tile of queries
    ((3, 6), 250, 300, 40, False, 8.0),      # head columns in no sixteens: one tile
    ((2, 3), 50, 120, 64, True, 4.0),
    ((5,), 70, 200, 48, False, 8.0),         # V's columns one by one, in all its forms
    ((2, 3), 33, 200, 40, True, 8.0),
    ((5,), 70, 333, 32, True, 8.0),
    ((3,), 20, 270, 16, True, 8.0),
])
@pytest.mark.parametrize("masked,where", [(False, False), (True, False), (False, True), (True, True)], ids=["plain", "mask", "cond", "both"])
def test_attention_pairs(device, batch, sq, skv, d, turned, divisor, masked, where):
    got, want = run(device, batch, sq, skv, d, masked, where, turned, divisor)
    # scores up to d / divisor with an error of d roundings each, weights that sum to one, values up to one
    assert (got - want).abs().max() <= 2.0 ** -24 * (2 * d * d / divisor / 4 + skv / 16 + 16)


def test_attention_pairs_not_finite(device):
    """A NaN in one query reaches its row alone, keys masked by -inf reach none, an infinity in V its column."""
    import torch

    got, want = run(device, (17,), 256, 512, 64, True, False, False, 8.0, spoil=True)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    fine = want.isfinite()
    assert (got - want)[fine].abs().max() <= 2.0 ** -24 * (2 * 64 * 64 / 8 / 4 + 512 / 16 + 16)


@pytest.mark.parametrize("d,skv", [(40, 200), (64, 256), (32, 300)])
@pytest.mark.parametrize("masked,where", [(False, False), (True, False), (False, True), (True, True)], ids=["plain", "mask", "cond", "both"])
def test_attention_scattered_fits(device, d, skv, masked, where):
    """V in columns one by one: up to 256 keys, beyond with up to 32 head columns, two workgroups fit a compute unit."""
    import torch

    from util import launches

    t = torch.rand(2, d, skv, device=device)
    q, kt, v = torch.rand(2, 64, d, device=device), t, t.transpose(1, 2)
    mask = torch.rand(1, 1, skv, device=device) if masked else None
    cond = torch.ones(1, 64, skv, dtype=torch.bool, device=device) if where else None
    out = torch.empty(2, 64, d, device=device)

    def call(stream):
        from fluidml_amd import cabi

        cabi.call("attention", ref(q), ref(kt), ref(v), ref(out), ctypes.c_double(8.0), 1, ref(mask) if masked else None,
                  ref(cond) if where else None, ctypes.c_double(-1e9), stream)

    call(None)
    (name, fit), = launches(call)
    assert "AttentionKernel" in name and fit >= 2
