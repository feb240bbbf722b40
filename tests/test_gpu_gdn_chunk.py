"""GPU parity of the delta net's 16-token chunks (k_gdn_chunk, k_gdn_delta_chunk) at the
edges of a chunk, of the batches that take them and of the 16 value heads one block
takes at a time, with the last bin of beta and alpha part full, and with a token whose
values are not finite: nothing of it reaches the tokens before it or other rows of the
state.  Against the CPU restatement, within the 1e-3 of the reference's magnitude that
one rounding step of a re-quantized activation moves an output by; the state, that no
quantization follows, within 2e-5: 128 products of sums of up to 33 fp32 terms (n eps
= 2e-6 each) over the restatement's float32 inputs."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from questwend_amd import ops  # noqa: E402
from oracle_lib import GdnWeights, Oracle, Q4_K, Q6_K, Q8_0, gdn_seg_restated  # noqa: E402
from test_gpu_attn import rel  # noqa: E402
from test_gpu_gdn import GpuGdn  # noqa: E402

TOL, STATE_TOL = 1e-3, 2e-5


@pytest.fixture(scope="module", autouse=True)
def lib_init():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    ops.init(0, 512 << 20)


@pytest.fixture(scope="module")
def orc():
    return Oracle()


@pytest.mark.parametrize("H_k,H_v,types", [(2, 4, (Q4_K, Q6_K, Q8_0, Q8_0, Q4_K)), (1, 17, (Q8_0,) * 5)])
@pytest.mark.parametrize("T", [31, 32, 33, 47, 64, 65, 129, 402])
def test_chunks(orc, H_k, H_v, types, T):
    gw = GdnWeights(512, 128, H_k, H_v, 4, types, 7 + T, orc)
    h = np.random.default_rng(T).standard_normal((T, 512)).astype(np.float32)
    cs, ss = gw.fresh_state(np.random.default_rng(5))
    g = GpuGdn(gw, cs, ss)
    got = g.run(h)
    want = gdn_seg_restated(gw, h, cs, ss, orc)
    gcs, gss = g.states()
    assert np.array_equal(gcs, cs)
    assert rel(got[0], want[0]) < TOL and rel(got[1], want[1]) < TOL
    assert rel(gss, ss) < STATE_TOL


@pytest.mark.parametrize("types", [(Q4_K, Q6_K, Q8_0, Q8_0, Q4_K), (Q8_0,) * 5])
@pytest.mark.parametrize("parts", [(1,) * 9, (1, 3, 8, 19), (4, 27), (7, 8, 9), (2, 29)])
def test_parts_give_the_same_bits(orc, types, parts):
    """Calls of fewer than 32 tokens: outputs and states bit for bit those of any parts."""
    T = sum(parts)
    gw = GdnWeights(512, 128, 2, 4, 4, types, 11, orc)
    h = np.random.default_rng(T).standard_normal((T, 512)).astype(np.float32)
    cs, ss = gw.fresh_state(np.random.default_rng(5))
    whole, split = GpuGdn(gw, cs, ss), GpuGdn(gw, cs, ss)
    want = whole.run(h)
    got = [split.run(p) for p in np.split(h, np.cumsum(parts)[:-1])]
    for i in range(2):
        assert np.array_equal(np.concatenate([g[i] for g in got]), want[i])
        assert np.array_equal(split.states()[i], whole.states()[i])


def test_ssm_norm_at_any_address(orc):
    gw = GdnWeights(512, 128, 2, 4, 4, (Q4_K, Q6_K, Q8_0, Q8_0, Q4_K), 12, orc)
    h = np.random.default_rng(1).standard_normal((5, 512)).astype(np.float32)
    cs, ss = gw.fresh_state(np.random.default_rng(5))
    want = GpuGdn(gw, cs, ss).run(h)
    g = GpuGdn(gw, cs, ss)
    off = torch.zeros(131, dtype=torch.float32, device="cuda:0")
    off[3:] = g.t[9]
    g.t[9] = off
    g.layer.ssm_norm = off.data_ptr() + 12
    got = g.run(h)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("T,p", [(40, 21), (32, 9), (37, 36)])
def test_overflow_stays_with_its_token(orc, T, p):
    """Value channel 3 of head 1: its projection reads only columns that are zero before
    token p, its current-token tap overflows there."""
    gw = GdnWeights(512, 128, 2, 4, 4, (Q4_K, Q6_K, Q8_0, Q8_0, Q4_K), 3, orc)
    c = 2 * gw.key_dim + 128 + 3
    rows = gw.w_qkv.reshape(gw.conv_ch, 288)
    rows[c, 144:] = 0
    gw.conv1d[c] = (0.0, 0.0, 0.0, 3e38)
    w = orc.dequantize(Q4_K, rows[c].copy(), 512).reshape(-1)
    h = np.random.default_rng(T).standard_normal((T, 512)).astype(np.float32)
    h[:p, :256] = 0.0
    h[p, :256] = 8.0 * np.sign(w[:256])
    cs, ss = gw.fresh_state(np.random.default_rng(5))
    g = GpuGdn(gw, cs, ss)
    got = g.run(h)
    with np.errstate(all="ignore"):
        gdn_seg_restated(gw, h, cs.copy(), s2 := ss.copy(), orc)
    want = gdn_seg_restated(gw, h[:p], cs, ss, orc)
    assert rel(got[0][:p], want[0]) < TOL and rel(got[1][:p], want[1]) < TOL
    gss = g.states()[1]
    assert not np.isfinite(gss[1, 3]).any() and not np.isfinite(s2[1, 3]).any()
    gss[1, 3] = s2[1, 3] = 0.0
    assert rel(gss, s2) < STATE_TOL
