"""GPU parity of the attention and delta-net halves at the edges of their tiles.

Attention (attn.hip): query rows around 32 and 64 (one, two and four waves), chunks
and splits of 64 keys around their ends, a first token without a past, heads per kv
head that do not divide 32, an odd number of heads (f32 attention output), one and
several PV splits.  Delta net (gdn.hip): tokens around the 4-token step, the 32
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
from questwend_amd import ops  # noqa: E402
from oracle_lib import (AttnWeights, GdnWeights, Oracle, Q4_K, Q6_K, Q8_0, attn_seg_restated,  # noqa: E402
                        gdn_seg_restated)
from test_gpu_attn import GpuAttn, dev, rel  # noqa: E402
from test_gpu_gdn import GpuGdn  # noqa: E402

TOL = 1e-3


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
