"""GPU parity of the weight quantizers and dequantizers (quantize.hip) where their
forms part: sub-blocks that the float search may not take (values so small or so
far apart that a scaled value leaves nearest_int's range), constant, all-zero and
one-sided sub-blocks, scales that round to 0, rows at addresses that allow no
16-byte access, and counts that do not fill a workgroup.  Bytes (and dequantized
floats) bit for bit against the CPU oracle."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from questwend_amd import check, lib, ops, row_size  # noqa: E402
from oracle_lib import Oracle, Q4_K, Q6_K, Q8_0  # noqa: E402
from test_gpu_parity import bits, dev, host  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def lib_init():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ops.init(0, 256 << 20)


@pytest.fixture(scope="module")
def orc():
    return Oracle()


def edge_values(rng, nblocks):
    """[nblocks, 256] with every 32-value sub-block of some kind."""
    x = (rng.standard_normal((nblocks * 8, 32)) * 0.02).astype(np.float32)
    for i in range(x.shape[0]):
        kind = i % 13
        if kind == 1:
            x[i] = 0.0
        elif kind == 2:
            x[i] = np.float32(0.013)                       # constant
        elif kind == 3:
            x[i] = -np.abs(x[i])                           # one-sided
        elif kind == 4:
            x[i] = np.abs(x[i]) + np.float32(0.5)
        elif kind == 5:
            x[i] *= np.float32(1e-30)                      # scale rounds to 0 beside its neighbours
        elif kind == 6:
            x[i] *= np.float32(1e-37)                      # denormal range
        elif kind == 7:
            x[i] = np.round(x[i] * 400) / np.float32(400)  # many ties
        elif kind == 8:
            x[i, 1:] = x[i, 0]
            x[i, 17] = np.nextafter(x[i, 0], np.float32(1))   # two neighbouring values: iscale huge
        elif kind == 9:
            x[i, 5] = np.float32(3e4)                      # one outlier
        elif kind == 10:
            x[i] *= np.float32(1e-14)                      # below and around Q6_K's 1e-15 bar
    return x.reshape(nblocks, 256)


@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q8_0])
@pytest.mark.parametrize("nblocks", [1, 33, 1300])
def test_quantize_edges(orc, t, nblocks):
    x = edge_values(np.random.default_rng(nblocks), nblocks)
    if t == Q8_0:   # (1 / d overflows in the reference for values this small, and its cast of inf is undefined)
        x[np.abs(x) < 1e-30] = 0.0
    assert np.array_equal(host(ops.quantize_chunk(t, dev(x))).reshape(-1), orc.quantize(t, x))


@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q8_0])
@pytest.mark.parametrize("so,do", [(1, 0), (0, 1), (2, 2), (0, 4)])
def test_unaligned(orc, t, so, do):
    """src so floats, dst (and the blocks read back) do bytes, y so floats past an aligned address."""
    n, blocks = 256 * 9, 9
    x = edge_values(np.random.default_rng(7), blocks).reshape(-1)
    if t == Q8_0:
        x[np.abs(x) < 1e-30] = 0.0
    src = torch.zeros(n + 8, dtype=torch.float32, device="cuda:0")
    src[so:so + n] = dev(x)
    want = orc.quantize(t, x)
    dst = torch.zeros(want.size + 16, dtype=torch.uint8, device="cuda:0")
    check(lib().qwmoe_quantize_chunk(ops.stream(), t, src.data_ptr() + 4 * so, dst.data_ptr() + do, blocks, 256))
    assert row_size(t, 256) * blocks == want.size
    assert np.array_equal(host(dst)[do:do + want.size], want)
    assert not host(dst)[do + want.size:].any() and not host(dst)[:do].any()
    if t != Q8_0 or do % 2 == 0:
        y = torch.zeros(n + 8, dtype=torch.float32, device="cuda:0")
        check(lib().qwmoe_dequantize(ops.stream(), t, dst.data_ptr() + do, y.data_ptr() + 4 * so, n))
        assert np.array_equal(bits(host(y)[so:so + n]), bits(orc.dequantize(t, want, n)))
