"""The row filter's candidate lists at the edges of its sorts: 1 .. 64, .. 256,
.. 512 and more entries, for top-k (candidates at or above the k-th largest chunk
maximum) and for top-p (ties of the boundary value, whose order is the index's).
Kept sets, probabilities and tokens bit for bit against the CPU oracle, which
evaluates the same arithmetic."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = (1, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300, 511, 512, 513, 700)


def _check(hv, orc, cuda, x, T, K, P, seed):
    u = np.random.default_rng(seed).random(len(x), dtype=np.float32)
    dev = [torch.from_numpy(a).to(cuda) for a in (T, K, P)]
    r = hv.ops.sample_rows(torch.from_numpy(x).to(cuda), *dev, mode="filtered",
                           uniforms=torch.from_numpy(u).to(cuda), want_probs=True)
    ref = orc.sampler(x, T, K, P, mode="filtered", uniforms=u)
    np.testing.assert_array_equal(r["probs"].cpu().numpy(), ref["probs"])
    np.testing.assert_array_equal(r["tokens"].cpu().numpy(), ref["tokens"])


@pytest.mark.parametrize("top_p", [1.0, 0.85])
def test_top_k_list_lengths(hv, orc, cuda, top_p):
    """One chunk holds n large values and every other one a single such value, so
    n + 19 candidates reach the 20th largest chunk maximum or fewer."""
    rng = np.random.default_rng(11)
    V, k = 40 * 2048, 20
    x = rng.standard_normal((len(SIZES), V)).astype(np.float32)
    for row, n in zip(x, SIZES):
        at = rng.permutation(2048)[:n]
        row[at] = 12.0 + rng.permutation(n).astype(np.float32) / 1024
        row[2048 * np.arange(1, k) + 5] = 10.0 + rng.random(k - 1).astype(np.float32)
    B = len(x)
    _check(hv, orc, cuda, x, np.full(B, 0.9, np.float32), np.full(B, k, np.int32),
           np.full(B, top_p, np.float32), 1)


@pytest.mark.parametrize("others", [0, 400])
def test_top_p_ties(hv, orc, cuda, others):
    """n ties carry the crossing; with `others` more elements in their coarse bucket
    the boundary sub-bucket is picked from the listed bucket."""
    rng = np.random.default_rng(12)
    V = 3 * 2048
    x = rng.standard_normal((len(SIZES), V)).astype(np.float32) - 20.0
    for row, n in zip(x, SIZES):
        at = rng.permutation(V)[:n + others]
        row[at[:n]] = 2.0
        row[at[n:]] = 2.0 + 0.05 * rng.random(others).astype(np.float32) + 0.01
        row[at[0]] = 3.03
    B = len(x)
    for p in (0.3, 0.9):
        _check(hv, orc, cuda, x, np.ones(B, np.float32), np.zeros(B, np.int32),
               np.full(B, p, np.float32), 2)


@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("ties", [False, True])
def test_top_p_long_buckets(hv, orc, cuda, ties, aligned):
    """Coarse buckets around the list's 8192 entries, of distinct values or all one
    value (more ties than the row filter's LDS holds), for both passes (the second
    needs rows of a multiple of 8)."""
    rng = np.random.default_rng(13)
    V = 9 * 2048 if aligned else 9 * 2048 + 3
    x = rng.standard_normal((7, V)).astype(np.float32) - 20.0
    for row, n in zip(x, (257, 4095, 4096, 4097, 8191, 8192, 8193)):
        at = rng.permutation(V)[:n]
        row[at] = 2.0 if ties else 2.0 + 0.12 * rng.random(n).astype(np.float32)
        row[at[0]] = 2.124
    B = len(x)
    for p in (0.4, 0.95):
        _check(hv, orc, cuda, x, np.ones(B, np.float32), np.zeros(B, np.int32),
               np.full(B, p, np.float32), 3)
