"""GPU parity of the persistent matrix-core kernel (k_mmid_mfma_hp) on block bytes
of the whole range -- every quant, every 6-bit or int8 scale, extreme activations
-- bit for bit against the CPU oracle: Q4_K and Q6_K, row lengths whose Q6_K rows
start on and off a dword, one- and two-tile items of every remainder, launches small
enough for 16-row items and large enough for 32-row ones, light bins in more 16-row
units than workgroups.  The dense cases send every bin to the matrix cores whatever
the row threshold; the sparse ones at the end split the bins between the GEMV and the
matrix cores (mul_mat_id, and whole layers, whose quantizing launches write the f16 copy)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from questwend_amd import ops  # noqa: E402
from oracle_lib import LayerWeights, Oracle, Q4_K, Q6_K, Q8_0  # noqa: E402
from test_gpu_parity import _layer_gpu, bits, dev, host  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def lib_init():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ops.init(0, 512 << 20)


@pytest.fixture(scope="module")
def orc():
    return Oracle()


def raw_blocks(rng, t, rows, K):
    nb = K // 256
    size, d_at = (144, 0) if t == Q4_K else (210, 208)
    w = rng.integers(0, 256, (rows, nb, size)).astype(np.uint8)
    d = (rng.standard_normal((rows, nb, 2 if t == Q4_K else 1)) * 1e-3).astype(np.float16)
    w[..., d_at:d_at + 2 * d.shape[-1]] = d.view(np.uint8).reshape(rows, nb, -1)
    if t == Q6_K:
        w[0, :, 192:208] = 0x80          # scales all -128 ...
        w[0, :, 0:192] = 0xff            # ... times quants all 63
        w[1, :, 192:208] = 0x7f
    else:
        w[0, :, 4:] = 0xff
    return w.reshape(-1)


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("K,N", [(768, 64), (1024, 192), (2048, 64), (2816, 128)])
@pytest.mark.parametrize("min_rows", [1, 8])
@pytest.mark.parametrize("many", [False, True])
def test_raw_blocks(orc, t, K, N, min_rows, many):
    rng = np.random.default_rng(K + N + min_rows)
    counts = [1, 8, 15, 16, 17, 31, 32, 33, 48, 49, 7, 64]
    if many:   # enough units for 32-row items: every expert again, four times over
        counts = counts * (4 if N > 64 else 8)
    n_as = len(counts)
    w = raw_blocks(rng, t, n_as * N, K)
    ids = rng.permutation(np.repeat(np.arange(n_as), counts)).astype(np.int32).reshape(-1, 1)
    b = rng.standard_normal((ids.shape[0], 1, K)).astype(np.float32)
    b[0] = np.float32(3.0)               # a row of equal values: quants all -127
    b[1, 0, 256:512] = 0.0
    prev = ops.set_mfma_min_rows(min_rows)
    try:
        got = host(ops.mul_mat_id(t, dev(w), K, N, n_as, dev(b), dev(ids)))
    finally:
        ops.set_mfma_min_rows(prev)
    assert np.array_equal(bits(got), bits(orc.mul_mat_id(t, K, N, n_as, w, b, ids)))


@pytest.mark.parametrize("t", [Q4_K, Q6_K])
@pytest.mark.parametrize("min_rows,per_bin", [(1, 13), (1, 14), (8, 13)])
def test_light_bins(orc, t, min_rows, per_bin):
    """The line of the 16-row items, 13 rows per bin, with more units (16 tiles of 64 weight
    rows per item) than the 768 workgroups, so that they walk from unit to unit."""
    K, N, n_as = 768, 1024, 48
    rng = np.random.default_rng(per_bin + min_rows)
    counts = np.tile([1, 16, 17, 33, 2, 9], n_as // 6)   # 13 per bin
    counts[0] += (per_bin - 13) * n_as
    w = raw_blocks(rng, t, n_as * N, K)
    ids = rng.permutation(np.repeat(np.arange(n_as), counts)).astype(np.int32).reshape(-1, 1)
    b = rng.standard_normal((ids.shape[0], 1, K)).astype(np.float32)
    prev = ops.set_mfma_min_rows(min_rows)
    try:
        got = host(ops.mul_mat_id(t, dev(w), K, N, n_as, dev(b), dev(ids)))
    finally:
        ops.set_mfma_min_rows(prev)
    assert np.array_equal(bits(got), bits(orc.mul_mat_id(t, K, N, n_as, w, b, ids)))


SPARSE = [9, 17, 33, 8, 1, 2, 3, 4, 5, 6, 7]   # 95 rows: four bins for the matrix cores, the rest the GEMV's


# bins: more than the rows' density asks for, so that the light ones stay on the GEMV
@pytest.mark.parametrize("t,n_as", [(Q4_K, 200), (Q4_K, 256), (Q6_K, 32), (Q6_K, 200), (Q8_0, 64), (Q8_0, 200)])
@pytest.mark.parametrize("K,N", [(768, 64), (2048, 128)])
def test_sparse_bins(orc, t, n_as, K, N):
    rng = np.random.default_rng(K + n_as)
    counts = np.zeros(n_as, np.int64)
    counts[rng.permutation(n_as)[:len(SPARSE)]] = SPARSE
    if t == Q8_0:
        w = orc.quantize(t, (rng.standard_normal((n_as * N, K)) * 0.02).astype(np.float32))
    else:
        w = raw_blocks(rng, t, n_as * N, K)
    ids = rng.permutation(np.repeat(np.arange(n_as), counts)).astype(np.int32).reshape(-1, 1)
    b = rng.standard_normal((ids.shape[0], 1, K)).astype(np.float32)
    prev = ops.set_mfma_min_rows(8)
    try:
        got = host(ops.mul_mat_id(t, dev(w), K, N, n_as, dev(b), dev(ids)))
    finally:
        ops.set_mfma_min_rows(prev)
    assert np.array_equal(bits(got), bits(orc.mul_mat_id(t, K, N, n_as, w, b, ids)))


@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q8_0])
@pytest.mark.parametrize("permute", [False, True])
def test_sparse_layer(orc, t, permute):
    """36 tokens over 80 experts, one each: 17 on expert 3, 9 on expert 9, the rest as the router has it."""
    H = F = 768
    E, T = 80, 36
    rng = np.random.default_rng(4)
    lw = LayerWeights.__new__(LayerWeights)
    lw.H, lw.E, lw.k, lw.F, lw.n_slots = H, E, 1, F, E
    lw.type_gate = lw.type_up = lw.type_down = t
    lw.slot_of = tuple(rng.permutation(E).astype(np.int32) for _ in range(3)) if permute else None
    def raw():
        if t != Q8_0:
            return raw_blocks(rng, t, E * H, F)
        w = rng.integers(0, 256, (E * H * F // 32, 34)).astype(np.uint8)
        w[:, :2] = (rng.standard_normal((w.shape[0], 1)) * 1e-3).astype(np.float16).view(np.uint8)
        return w.reshape(-1)
    lw.gate, lw.up, lw.down = raw(), raw(), raw()
    lw.router = (rng.standard_normal((E, H)) * 0.02).astype(np.float32)
    x = rng.standard_normal((T, H)).astype(np.float32)
    x[:, :2] = 0.0
    x[:17, 0] = x[17:26, 1] = 3.0
    lw.router[3, 0] = lw.router[9, 1] = 20.0
    prev, form = ops.set_mfma_min_rows(8), ops.set_mfma_form(ops.MFMA_EXACT)
    try:
        L, keep, _ = _layer_gpu(lw)
        out, xn, ids, w = ops.ffn_layer(L, dev(x), 1e-6)
        out, ids = host(out), host(ids)
    finally:
        ops.set_mfma_min_rows(prev)
        ops.set_mfma_form(form)
    r = orc.moe_layer(lw, x, rms_eps=1e-6)
    n = np.bincount(ids.reshape(-1), minlength=E)
    assert n[3] >= 17 and n[9] >= 9 and (n > 0).sum() > 6 and np.sort(n)[-3] < 8
    assert np.array_equal(ids, r["ids"]) and np.array_equal(bits(out), bits(r["out"]))
