"""GPU parity of the attention and delta-net halves at the edges of their tiles.

Attention (attn.hip): query rows around 32 and 64 (one, two and four waves), chunks
and splits of 64 keys around their ends, a first token without a past, heads per kv
head that do not divide 32, an odd number of heads (f32 attention output), one and
several PV splits, as a small workspace has them (merged, the last group ragged), and the
smallest workspace that a call fits.  Delta net (gdn.hip): tokens around the 4-token step, the 32
tokens from which it takes 16 at a time and the ends of those chunks, every
number of conv taps, an odd number of value heads, Q8_0 throughout.

Against the CPU restatements (oracle_lib, pinned to ggml), within the 1e-3 of the
reference's magnitude that a rounding step of a re-quantized activation or an f16
probability moves an output by; copies of projection outputs bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from questwend_amd import QwmoeError, ops, row_size, vec_dot_type  # noqa: E402
from oracle_lib import (AttnWeights, GdnWeights, Oracle, Q4_K, Q6_K, Q8_0, attn_seg_restated,  # noqa: E402
                        gdn_seg_restated)
from test_gpu_attn import GpuAttn, dev, rel  # noqa: E402
from test_gpu_gdn import GpuGdn  # noqa: E402

TOL = 1e-3
ERR_WORKSPACE = -4


@pytest.fixture(scope="module", autouse=True)
def lib_init():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ops.init(0, 512 << 20)


@pytest.fixture(scope="module")
def orc():
    return Oracle()


def attn_case(orc, heads, types, T, n_past, seed=1):
    nq, nk = heads
    aw = AttnWeights(512, nq, nk, 128, types, seed=seed, oracle=orc)
    rng = np.random.default_rng(T + n_past)
    n_ctx = n_past + T + 3
    kc = np.full((n_ctx, nk * 128), 0x7e00, np.uint16)   # NaN past the cached rows: never to be read
    vc = kc.copy()
    for c in (kc, vc):
        c[:n_past] = (rng.standard_normal((n_past, nk * 128)) * 0.5).astype(np.float16).view(np.uint16)
    h = rng.standard_normal((T, 512)).astype(np.float32)
    g = GpuAttn(aw, n_ctx, kc, vc)
    res, fin = ops.attn_seg(g.layer, dev(h), n_past)
    torch.cuda.synchronize()
    kr, vr = kc.copy(), vc.copy()
    want_res, want_fin, _, _ = attn_seg_restated(aw, h, n_past, kr, vr, orc)
    assert rel(res.cpu().numpy(), want_res) < TOL and rel(fin.cpu().numpy(), want_fin) < TOL
    assert np.array_equal(g.caches()[1], vr)


@pytest.mark.parametrize("T,n_past", [(1, 0), (1, 63), (1, 64), (8, 56), (9, 120), (16, 0), (17, 47), (33, 31), (2, 1000)])
def test_attention(orc, T, n_past):
    attn_case(orc, (8, 2), (Q4_K, Q4_K, Q6_K, Q4_K), T, n_past)


@pytest.mark.parametrize("T,n_past", [(1, 5), (11, 60), (22, 128), (50, 300)])
def test_attention_odd_heads(orc, T, n_past):
    attn_case(orc, (3, 1), (Q8_0,) * 4, T, n_past)


@pytest.mark.parametrize("T", [4096, 4])
def test_attention_long_sum(orc, T):
    """The softmax's sum over 100 k keys of which one holds nearly everything: each of the
    others adds 0.9 * 2^-28, a group of sixteen less than half a step of a 32-bit 1.0.  All
    together they take that one's probability below 1 - 2^-12, the middle between the f16s 1
    and 1 - 2^-11; with those beside the largest key lost, it is above.  T = 4096: one split
    over all keys.  The query turns with its position in a pair of dims that the rotary
    base leaves still, so every row has the same result: that of the CPU restatement, whose
    sum is in double, within 1e-5 (a step of p is 5e-4)."""
    n = 100096
    aw = AttnWeights(512, 16, 1, 128, (Q4_K, Q4_K, Q8_0, Q4_K), seed=3, oracle=orc, freq_base=1e38)
    aw.wq = np.ascontiguousarray(np.tile(aw.wq.reshape(16, -1)[:1], (16, 1)).reshape(-1))   # every head the same query
    aw.k_norm[:] = 0.0                                                                      # new keys: score 0
    keep = aw.q_norm[[63, 127]].copy()
    aw.q_norm[:] = 0.0
    aw.q_norm[[63, 127]] = 10.0 * keep
    h = np.random.default_rng(8).standard_normal((1, 512)).astype(np.float32)
    kc, vc = np.zeros((n, 128), np.uint16), np.zeros((n, 128), np.uint16)
    q = attn_seg_restated(aw, h, 1, kc[:2].copy(), vc[:2].copy(), orc)[2][0, :128].astype(np.float16).astype(np.float64)
    s = 28.0 * np.log(2.0) - np.log(0.9)
    kc[0] = (q * (s * np.sqrt(128.0) / (q @ q))).astype(np.float16).view(np.uint16)
    vc[0] = np.random.default_rng(9).standard_normal(128).astype(np.float16).view(np.uint16)
    g = GpuAttn(aw, n, kc, vc)
    res, _ = ops.attn_seg(g.layer, dev(np.repeat(h, T, 0)), n - T)
    want, _, _, att = attn_seg_restated(aw, h, n - 1, kc.copy(), vc.copy(), orc)
    v0 = vc[0].view(np.float16).astype(np.float32)
    assert np.allclose(att.reshape(16, 128), (1.0 - 2.0 ** -11) * v0, rtol=1e-6, atol=0)   # (p is where it should be)
    got = res.cpu().numpy() - h
    assert rel(got, np.repeat(want - h, T, 0)) < 1e-5


@pytest.mark.parametrize("heads,types,T,n_past", [((8, 2), (Q4_K, Q4_K, Q6_K, Q4_K), 3, 1000), ((3, 1), (Q8_0,) * 4, 2, 700),
                                                  ((8, 1), (Q4_K,) * 4, 32, 16082)])
def test_attention_workspaces(orc, heads, types, T, n_past):
    """From the smallest workspace that the call fits (which the header states) up, one PV
    split at a time: 1, 2, 3 ... of the statistics' splits together."""
    nq, nk = heads
    H, NQ, NK = 512, nq * 128, nk * 128
    aw = AttnWeights(H, nq, nk, 128, types, seed=2, oracle=orc)
    rng = np.random.default_rng(T + n_past)
    kc = np.full((n_past + T, NK), 0x7e00, np.uint16)
    vc = kc.copy()
    for c in (kc, vc):
        c[:n_past] = (rng.standard_normal((n_past, NK)) * 0.5).astype(np.float16).view(np.uint16)
    h = rng.standard_normal((T, H)).astype(np.float32)
    kr, vr = kc.copy(), vc.copy()
    want = attn_seg_restated(aw, h, n_past, kr, vr, orc)[:2]
    hd = dev(h)

    def call(size):
        """Whether a workspace of `size` bytes takes the call; the result checked, or that nothing was written."""
        g = GpuAttn(aw, n_past + T, kc, vc)
        ops.shutdown()
        ops.init(0, size)
        try:
            got = ops.attn_seg(g.layer, hd, n_past)
        except QwmoeError as e:
            assert e.status == ERR_WORKSPACE
            torch.cuda.synchronize()
            assert np.array_equal(g.caches()[1], vc)
            return False
        torch.cuda.synchronize()
        assert rel(got[0].cpu().numpy(), want[0]) < TOL and rel(got[1].cpu().numpy(), want[1]) < TOL
        assert np.array_equal(g.caches()[1], vr)
        return True

    per_pv = 4 * T * NQ
    quantized = sum(row_size(vec_dot_type(t), n) for t, n in ((types[0], H), (types[3], NQ)))
    least = T * (4 * (NQ + 2 * NK + H) + (4 * H if Q8_0 in types else 0) + 2 * NQ + quantized + 8 * nq) + per_pv
    try:
        lo, hi = 4096, least + 16384   # (alignment of some twenty buffers)
        assert call(hi) and not call(lo)
        while hi - lo > 256:
            mid = (lo + hi) // 512 * 256
            lo, hi = (lo, mid) if call(mid) else (mid, hi)
        beside = 17 * T * (H + NQ) // 8 + per_pv + 8192
        for i in range(min(18, (n_past + T) // 64 + 2) if T < 32 else 4):
            assert call(hi + beside + i * per_pv)
    finally:
        ops.shutdown()
        ops.init(0, 512 << 20)


def gdn_case(orc, H_k, H_v, d_conv, types, T):
    gw = GdnWeights(512, 128, H_k, H_v, d_conv, types, 7 + T, orc)
    h = np.random.default_rng(T).standard_normal((T, 512)).astype(np.float32)
    cs, ss = gw.fresh_state(np.random.default_rng(5))
    g = GpuGdn(gw, cs, ss)
    got = g.run(h)
    want = gdn_seg_restated(gw, h, cs, ss, orc)
    gcs, gss = g.states()
    assert np.array_equal(gcs, cs)
    assert rel(got[0], want[0]) < TOL and rel(got[1], want[1]) < TOL and rel(gss, ss) < TOL


@pytest.mark.parametrize("T", [2, 3, 4, 31, 32, 33, 63, 66])
def test_delta_net(orc, T):
    gdn_case(orc, 2, 4, 4, (Q4_K, Q6_K, Q8_0, Q8_0, Q4_K), T)


@pytest.mark.parametrize("d_conv", [2, 3, 5, 6, 7, 8])
def test_delta_net_taps(orc, d_conv):
    gdn_case(orc, 1, 3, d_conv, (Q8_0,) * 5, 9)
