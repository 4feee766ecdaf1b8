"""Arguments that the C entry points refuse before anything is launched (no GPU: the addresses are never read)."""
import ctypes

import pytest

FL_ERR_SHAPE = -3
HERE = ctypes.create_string_buffer(4096)


@pytest.fixture
def cabi():
    import torch  # noqa: F401  (before fluidml_amd: the process then has one HIP runtime)
    from fluidml_amd import cabi

    return cabi


def tensor(cabi, *shape):
    base = (ctypes.addressof(HERE) + 255) // 256 * 256
    return cabi.make_tensor(base, cabi.FL_FLOAT32, shape)


@pytest.mark.parametrize("size,pads,out", [
    ((13, 15), (1, 1, 1, 1), (7, 8)),    # what stride 2 leaves
    ((13, 15), (2, 2, 2, 2), (13, 15)),  # what dilation 2 leaves
    ((13, 15), (0, 0, 0, 0), (11, 12)),
    ((13, 15), (0, 0, 0, 0), (12, 13)),
])
def test_packed_convolution_has_one_output_size(cabi, size, pads, out):
    x, w, o = tensor(cabi, 1, 32, *size), tensor(cabi, 32, 32, 3, 3), tensor(cabi, 1, 32, *out)
    rc = cabi.lib.fluidml_hip_conv3x3_packed_chain(ctypes.byref(x), ctypes.byref(w), x.base, 3, None, ctypes.byref(o),
                                                   cabi.i64_array(pads), None, 0, None)
    assert rc == FL_ERR_SHAPE


@pytest.mark.parametrize("rows,K,N", [
    (128, 768, 3072), (192, 768, 3072), (512, 768, 768),  # a twentieth faster, for half as much memory again
    (64, 4096, 4096), (20, 512, 50304),                   # slower
    (256, 3072, 768), (320, 3072, 768), (128, 2048, 2048),
])
def test_weights_not_worth_packing(cabi, rows, K, N):
    w, packed, size = tensor(cabi, K, N), ctypes.c_void_p(), ctypes.c_size_t()
    rc = cabi.lib.fluidml_hip_contract_pack(ctypes.byref(w), 0, rows, 3, None, ctypes.byref(packed), ctypes.byref(size))
    assert rc == cabi.FL_ERR_UNSUPPORTED and not packed.value
