"""Resampling and probabilities of filtered rows, at the edges of the kept-element
lists: chunks with none, one, 512 (the list's size), 513 and all elements kept,
vocabularies around one 2048-element chunk, output over the input. Bit for bit
against the CPU oracle, which evaluates the same arithmetic."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(hv, rng, V, dtype):
    """The last n places of a row hold its n largest values, and top-k keeps
    exactly those (n = V: nothing is filtered)."""
    T, K, P, x = [], [], [], []
    for n in (1, 2, 511, 512, 513, V):
        n = min(n, V)
        row = rng.standard_normal(V).astype(np.float32)
        row[V - n:] = 6.0 + rng.random(n).astype(np.float32)
        x.append(row)
        T.append(0.5 + rng.random())
        K.append(n if n < V else 0)
        P.append(1.0 if n != 512 else 0.95)
    x = np.stack(x)
    if dtype == "bf16":
        x = hv.synthetic.bf16_bits_to_f32(hv.synthetic.f32_to_bf16_bits(x))
    return x, np.array(T, np.float32), np.array(K, np.int32), np.array(P, np.float32)


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
@pytest.mark.parametrize("V", [8, 2040, 2048, 2056, 4104, 6144])
def test_kept_lists_vs_oracle(hv, orc, cuda, V, dtype):
    rng = np.random.default_rng(V)
    x, T, K, P = _rows(hv, rng, V, dtype)
    lg = torch.from_numpy(x).to(cuda)
    if dtype == "bf16":
        lg = lg.to(torch.bfloat16)
    u = rng.random(len(x), dtype=np.float32)
    dev = [torch.from_numpy(a).to(cuda) for a in (T, K, P)]
    r = hv.ops.sample_rows(lg, *dev, mode="filtered", uniforms=torch.from_numpy(u).to(cuda),
                           want_probs=True)
    m = hv.ops.sample_rows(lg, *dev, mode="filtered", want_probs=True, out_kind=1)
    ref = orc.sampler(x, T, K, P, mode="filtered", uniforms=u)
    np.testing.assert_array_equal(r["probs"].cpu().numpy(), ref["probs"])
    np.testing.assert_array_equal(r["tokens"].cpu().numpy(), ref["tokens"])
    masked = m["probs"].cpu().numpy()
    xs = (x / T[:, None]).astype(np.float32)
    np.testing.assert_array_equal(masked, np.where(ref["probs"] > 0, xs, -np.inf))
    if dtype == "f32":  # probabilities written over the logits
        buf = lg.clone()
        hv.ops.sample_rows(buf, *dev, mode="filtered", probs_out=buf)
        np.testing.assert_array_equal(buf.cpu().numpy(), ref["probs"])


@pytest.mark.parametrize("V", [2040, 4104])
def test_kept_residual_vs_oracle(hv, orc, cuda, V):
    """Rejections at each position: the residual max(p - q, 0) over the lists."""
    rng = np.random.default_rng(V + 1)
    x, T, K, P = _rows(hv, rng, V, "bf16")
    B, R = len(x), 3
    x = np.ascontiguousarray(np.repeat(x[:, None], R, axis=1))
    q = rng.random((B, R - 1, V), dtype=np.float32)
    q /= q.sum(-1, keepdims=True)
    d = rng.integers(0, V, (B, R - 1))
    d[::2, 0] = V - 1  # a kept token: may be accepted
    ua = rng.random((B, R - 1), dtype=np.float32)
    ur = rng.random(B, dtype=np.float32)
    t = [torch.from_numpy(a).to(cuda) for a in (q, d, T, ua, ur, K, P)]
    nacc, out, olen = hv.ops.spec_accept(
        torch.from_numpy(x).to(cuda).to(torch.bfloat16), *t[:5], mode="filtered",
        top_ks=t[5], top_ps=t[6])[:3]
    ref = orc.spec_accept(x, q, d, T, ua, ur, mode="filtered", top_ks=K, top_ps=P)
    np.testing.assert_array_equal(nacc.cpu().numpy(), ref["num_accepted"])
    np.testing.assert_array_equal(out.cpu().numpy(), ref["out_tokens"])
    np.testing.assert_array_equal(olen.cpu().numpy(), ref["out_len"])


@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_kept_lists_with_subnormal_quotients(hv, orc, cuda, dtype):
    """A temperature so large that the logits over it are a few of the smallest subnormal:
    logits well below the boundary's share its rounded quotient and are kept with it."""
    rng = np.random.default_rng(3)
    V, tiny = 4104, 2.0 ** -149
    T = np.array([1e30, 3e33, 2.5e20], np.float32)
    x = (4.55 + 0.4 * rng.random((3, V))) * (tiny * T.astype(np.float64))[:, None]
    x[:, 2000:] = -x[:, 2000:]
    x = x.astype(np.float32)
    if dtype == "bf16":
        x = hv.synthetic.bf16_bits_to_f32(hv.synthetic.f32_to_bf16_bits(x))
    K, P = np.array([40, 700, 0], np.int32), np.array([1.0, 1.0, 0.3], np.float32)
    lg = torch.from_numpy(x).to(cuda)
    u = rng.random(3, dtype=np.float32)
    dev = [torch.from_numpy(a).to(cuda) for a in (T, K, P)]
    r = hv.ops.sample_rows(lg.to(torch.bfloat16) if dtype == "bf16" else lg, *dev, mode="filtered",
                           uniforms=torch.from_numpy(u).to(cuda), want_probs=True)
    ref = orc.sampler(x, T, K, P, mode="filtered", uniforms=u)
    np.testing.assert_array_equal(r["probs"].cpu().numpy(), ref["probs"])
    np.testing.assert_array_equal(r["tokens"].cpu().numpy(), ref["tokens"])
