"""GPU parity of the small-batch layer launches: top-k and grouping in one launch
at the edges of its one-wave grouping (64, 128 pairs), of the batch it takes (16
tokens) and of the 64 ranks one wave pass covers, with and without tied
probabilities, and the router launch's Q8_K rows and f16 copies.  Bit for bit
against the CPU oracle."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import questwend_amd as qa  # noqa: E402
from questwend_amd import ops  # noqa: E402
from oracle_lib import LayerWeights, Oracle, Q4_K, Q6_K, Q8_0  # noqa: E402
from test_gpu_parity import _layer_gpu, bits, dev, host, note  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def lib_init():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ops.init(0, 512 << 20)


@pytest.fixture(scope="module")
def orc():
    return Oracle()


@pytest.mark.parametrize("E,k,T", [(16, 8, 8), (16, 5, 13), (16, 13, 5), (24, 8, 16), (16, 11, 12),
                                   (128, 127, 1), (128, 128, 1), (128, 65, 2), (8, 1, 16), (40, 8, 9)])
@pytest.mark.parametrize("ties", [False, True])
def test_small_batch_layer(orc, E, k, T, ties):
    note(f"small-batch layer E={E} k={k} T={T} ties={ties}")
    types = (Q8_0,) * 3 if T % 2 else (Q4_K, Q4_K, Q6_K)
    lw = LayerWeights(512, E, k, 256, *types, seed=E + k + T, oracle=orc, permute=bool(k & 1))
    if ties:
        lw.router[1::2] = lw.router[::2]     # equal in pairs: ties inside and across the k-th place
    L, keep, _ = _layer_gpu(lw)
    x = np.random.default_rng(T).standard_normal((T, 512)).astype(np.float32)
    ops.device_status(clear=True)
    out, xn, ids, w = ops.ffn_layer(L, dev(x), rms_eps=1e-6)
    r = orc.moe_layer(lw, x, rms_eps=1e-6)
    assert np.array_equal(host(ids), r["ids"])
    assert np.array_equal(bits(host(w)), bits(r["weights"]))
    assert np.array_equal(bits(host(out)), bits(r["out"]))
    assert np.array_equal(bits(host(xn)), bits(r["xnext"]))
    assert ops.device_status(clear=True) == (qa.STATUS_TOPK_TIE_SORT if ties else 0)
