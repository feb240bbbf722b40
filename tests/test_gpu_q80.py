"""GPU parity of the Q8_0 mul_mat_id kernels (mmid_q80.hip): the matrix-core form
and the row-copying GEMV, bit for bit against the CPU oracle, at the edges of
their tiles: one row and full / partial 16-row items, weight rows that do
not fill a 16-row workgroup, the smallest and larger row lengths, each activation
row of a pass (1 to 4), the weights' extreme quants (-128), a workspace without
room for the f16 copy, a batch too sparse for it, and the SwiGLU launch that writes Q8_0
rows directly."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from questwend_amd import lib, ops  # noqa: E402
from oracle_lib import LayerWeights, Oracle, Q6_K, Q8_0, row_size, vec_dot_type  # noqa: E402
from test_gpu_decode import GpuLayer  # noqa: E402
from test_gpu_parity import bits, dev, host  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def lib_init():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ops.init(0, 512 << 20)
    prev = ops.set_mfma_min_rows(8)
    yield
    torch.cuda.synchronize()
    ops.set_mfma_min_rows(prev)


@pytest.fixture(scope="module")
def orc():
    return Oracle()


def counts_case(orc, K, N, counts, ne11, seed):
    """Expert a receives counts[a] of the (one-slot) rows; n_ids = ne11 slots."""
    rng = np.random.default_rng(seed)
    n_as = len(counts)
    w = orc.quantize(Q8_0, (rng.standard_normal((n_as * N, K)) * 0.02).astype(np.float32))
    w.reshape(-1, 34)[::7, 2 + seed % 32] = 0x80   # a quant of -128, which the quantizer never writes
    flat = rng.permutation(np.repeat(np.arange(n_as), counts)).astype(np.int32)
    ids = flat.reshape(-1, ne11)
    b = rng.standard_normal((ids.shape[0], ne11, K)).astype(np.float32)
    b[0, 0, :32] = 0.0   # a block of zeros (d = 0)
    want = orc.mul_mat_id(Q8_0, K, N, n_as, w, b, ids)
    return (lambda noalloc=False: host(ops.mul_mat_id(Q8_0, dev(w), K, N, n_as, dev(b), dev(ids), noalloc=noalloc))), want


@pytest.mark.parametrize("K,N", [(256, 64), (768, 128), (1280, 64), (2048, 192)])
@pytest.mark.parametrize("min_rows", [1, 8])
def test_matrix_cores(orc, K, N, min_rows):
    run, want = counts_case(orc, K, N, [1, 16, 17, 31, 32, 33, 65, 7, 0, 8], 2, seed=K + N)
    ops.set_mfma_min_rows(min_rows)
    try:
        assert np.array_equal(bits(run()), bits(want))
    finally:
        ops.set_mfma_min_rows(8)


def test_no_room_for_the_copy(orc):
    """The allocation-free call's 8 MiB hold the Q8_0 rows but not their f16 copy: the GEMV, the same bits."""
    run, want = counts_case(orc, 2048, 64, [900, 900], 1, seed=3)
    assert np.array_equal(bits(run(noalloc=True)), bits(want))


@pytest.mark.parametrize("t", [Q6_K, Q8_0])
def test_no_copy_that_nothing_reads(orc, t):
    """64 tokens, two of 512 experts each: the GEMV takes the bins, so the call's workspace holds the
    quantized rows and the grouping (under 100 KB) and no f16 copy of the rows (278 KB), nor is there a launch for it."""
    K, N, T, E = 2048, 64, 64, 512
    w = torch.zeros((E * N, row_size(t, K)), dtype=torch.uint8, device="cuda:0")
    b = torch.zeros((T, 1, K), dtype=torch.float32, device="cuda:0")
    ids = torch.arange(2 * T, dtype=torch.int32, device="cuda:0").view(T, 2)
    ops.shutdown()
    try:
        ops.init(0, 64 << 20)
        ops.mul_mat_id(t, w, K, N, E, b, ids)
        torch.cuda.synchronize()
        assert lib().qwmoe_workspace_high_water() < T * row_size(vec_dot_type(t), K) + 100_000
    finally:
        ops.init(0, 512 << 20)


@pytest.mark.parametrize("K", [256, 768, 2048, 4096, 64, 1088])
@pytest.mark.parametrize("N", [1, 8, 41])
def test_gemv(orc, K, N):
    run, want = counts_case(orc, K, N, [1, 2, 3, 4, 5, 7], 1, seed=K + N)
    assert np.array_equal(bits(run()), bits(want))


@pytest.mark.parametrize("T", [1, 3, 24])
def test_layer(orc, T):
    g = GpuLayer(1024, 16, 4, 320, (Q8_0,) * 3, seed=T)   # F = 320: down rows of the general GEMV
    x = np.random.default_rng(T).standard_normal((T, 1024)).astype(np.float32)
    out, xn, ids, w = ops.ffn_layer(g.layer, dev(x), 1e-6)
    r = orc.moe_layer(g.host, x, rms_eps=1e-6)
    assert np.array_equal(host(ids), r["ids"])
    assert np.array_equal(bits(host(out)), bits(r["out"]))
