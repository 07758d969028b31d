"""GPU parity of the prompt-sized query tiles (k_prefill_attn) with the float64
oracle: 128-row tiles over 64-key steps, at the edges of both. Outputs are bf16
and must agree within 2e-2 (absolute + relative), as the other attention tests."""
import numpy as np
import pytest
import torch

from test_gpu_attention import TOL, _bf16, _run, attn  # noqa: F401

pytestmark = pytest.mark.gpu


def _ragged(hv, lens_q, lens_k, hq, block_size, seed):
    w = hv.synthetic.attention_workload(batch=len(lens_k), q_len=max(lens_q), num_q_heads=hq,
                                        num_kv_heads=8, block_size=block_size, lens=lens_k,
                                        seed=seed)
    at = np.concatenate([[0], np.cumsum(np.minimum(max(lens_q), lens_k))])
    keep = np.concatenate([np.arange(at[b + 1] - n, at[b + 1]) for b, n in enumerate(lens_q)])
    w["q"] = np.ascontiguousarray(w["q"][keep])
    w["cu_seqlens_q"] = np.concatenate([[0], np.cumsum(lens_q)]).astype(np.int32)
    w["max_seqlen_q"] = int(max(lens_q))
    return w


# rows around one and two 128-row tiles, keys around the 64-key step, a one-token
# sequence beside long ones, cached prefixes that end inside a step; 4, 2, 1, 5, 8
# and 16 query heads per kv head; the smallest block, the default, one between
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("hq,block,lens_q,prefix", [
    (32, 256, [32, 31, 1, 17, 32, 30, 2, 32, 9, 32], 0),
    (32, 32, [33, 64, 63, 1, 65], [0, 31, 32, 200, 64]),
    (32, 64, [129, 128, 127], [1, 63, 65]),
    (16, 256, [257, 3, 191, 64, 255], [0, 300, 1, 256, 255]),
    (8, 128, [130, 513, 385], [0, 1, 127]),
    (40, 32, [52, 26, 51, 25, 77], 0),
    (64, 256, [100, 9, 31, 70], [0, 130, 64, 1]),
    (128, 256, [17, 40, 33], [0, 5, 300]),
])
def test_prefill_tiles(hv, attn, cuda, kv, hq, block, lens_q, prefix):  # noqa: F811
    print(f"prefill tiles {kv} hq={hq} block={block} q={lens_q} prefix={prefix}", flush=True)
    pre = [prefix] * len(lens_q) if isinstance(prefix, int) else prefix
    w = _ragged(hv, lens_q, [a + b for a, b in zip(lens_q, pre)], hq, block, sum(lens_q))
    _run(hv, attn, w, cuda, kv=kv, q_strided=hq == 32)


def test_prefill_skips_missing_blocks(hv, attn, cuda):  # noqa: F811
    """Keys whose block-table entry is no cache block are left out, as in the other
    launches: against the oracle over the remaining keys."""
    lens = [200] * 3
    w = hv.synthetic.attention_workload(batch=3, q_len=200, num_q_heads=32, num_kv_heads=8,
                                        block_size=32, lens=lens, seed=3)
    hole = [2, 3, 5]
    bt = w["block_tables"].copy()
    for b, e in enumerate(hole):
        bt[b, e] = -1 if b != 1 else 1 << 20
    out = hv.ops.verify_attention(
        _bf16(w["q"], cuda), _bf16(w["k_cache"], cuda), _bf16(w["v_cache"], cuda),
        torch.from_numpy(bt).to(cuda), torch.from_numpy(w["cu_seqlens_q"]).to(cuda),
        torch.from_numpy(w["cu_seqlens_k"]).to(cuda), 200, 200, w["softmax_scale"])
    got = out.float().cpu().numpy()
    for b, e in enumerate(hole):
        q = w["q"][200 * b:200 * b + 200]
        rest = np.delete(w["block_tables"][b], e)
        # queries past the hole: the same query over the keys without it
        late = np.arange(32 * (e + 1), 200)
        ref = attn.paged_attention(q[late], w["k_cache"], w["v_cache"], rest[None],
                                   np.array([0, late.size]), np.array([0, 168]),
                                   w["softmax_scale"])
        err = np.abs(got[200 * b + late] - ref)
        assert (err <= TOL + TOL * np.abs(ref)).all(), (b, err.max())


def test_prefill_unpaged_matches_paged(hv, cuda):
    """Unpaged rows and a paged cache holding them: the same bits."""
    lens = [150, 64, 129, 31]
    g = torch.Generator(device=cuda).manual_seed(5)
    n = sum(lens)
    q = torch.randn((n, 32, 128), generator=g, device=cuda).bfloat16()
    kv = torch.randn((n, 16, 128), generator=g, device=cuda).bfloat16()
    k, v = kv[:, :8], kv[:, 8:]
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=cuda)
    kc = torch.zeros((len(lens), 256, 8, 128), dtype=torch.bfloat16, device=cuda)
    vc = torch.zeros_like(kc)
    for b, m in enumerate(lens):
        kc[b, :m] = k[int(cu[b]):int(cu[b]) + m]
        vc[b, :m] = v[int(cu[b]):int(cu[b]) + m]
    bt = torch.arange(len(lens), dtype=torch.int32, device=cuda)[:, None].contiguous()
    a = hv.ops.verify_attention(q, k, v, None, cu, cu, 150, 150, 128 ** -0.5)
    b = hv.ops.verify_attention(q, kc, vc, bt, cu, cu, 150, 150, 128 ** -0.5)
    assert torch.equal(a, b)


# key splits: a few new tokens behind long prefixes beside a long prompt, prompts of
# few tiles behind prefixes just under, at and over a multiple of the shortest piece
# (1024 keys), block tables of more than 64 entries (one register of them), tiles that
# are one piece beside tiles that are several
@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("hq,block,lens_q,prefix", [
    (32, 256, [200, 1, 4, 1], [0, 3000, 1500, 2300]),
    (32, 32, [130, 129, 131], [2040, 4100, 2047]),
    (16, 64, [300, 2, 150], [5000, 1022, 0]),
    (8, 256, [700, 1], [1, 6000]),
])
def test_prefill_key_splits(hv, attn, cuda, kv, hq, block, lens_q, prefix):  # noqa: F811
    print(f"prefill splits {kv} hq={hq} block={block} q={lens_q} prefix={prefix}", flush=True)
    w = _ragged(hv, lens_q, [a + b for a, b in zip(lens_q, prefix)], hq, block, sum(lens_q))
    w["max_seqlen_k"] = max(w["max_seqlen_k"], 4096)
    _run(hv, attn, w, cuda, kv=kv)


def _call(hv, cuda, w, bt, kc, vc, declared):
    return hv.ops.verify_attention(
        _bf16(w["q"], cuda), kc, vc, torch.from_numpy(np.ascontiguousarray(bt)).to(cuda),
        torch.from_numpy(w["cu_seqlens_q"]).to(cuda), torch.from_numpy(w["cu_seqlens_k"]).to(cuda),
        w["max_seqlen_q"], declared, w["softmax_scale"])


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
def test_prefill_splits_skip_missing_blocks(hv, attn, cuda, kv):  # noqa: F811
    """Missing blocks beyond the first 64 table entries and in a piece of their own: the
    keys they hold are left out, against the oracle over the remaining keys; and the same
    call again gives the same bits, the merge counters left at zero."""
    lens_q, prefix = [130, 129, 131], [2944, 4100, 2047]
    w = _ragged(hv, lens_q, [a + b for a, b in zip(lens_q, prefix)], 32, 32, 7)
    hole = [70, 3, 40]
    bt = w["block_tables"].copy()
    for b, e in enumerate(hole):
        bt[b, e] = -1 if b else 1 << 20
    kc, vc = _bf16(w["k_cache"], cuda), _bf16(w["v_cache"], cuda)
    if kv == "fp8":
        kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    out = _call(hv, cuda, w, bt, kc, vc, 4608)
    assert torch.equal(out, _call(hv, cuda, w, bt, kc, vc, 4608))
    ws = hv.ops.workspace(cuda, 1, "attention")
    assert int(ws[:16384].view(torch.int32).abs().max()) == 0
    got = out.float().cpu().numpy()
    kd, vd = kc.float().cpu().numpy(), vc.float().cpu().numpy()
    for b, e in enumerate(hole):
        q0, q1 = int(w["cu_seqlens_q"][b]), int(w["cu_seqlens_q"][b + 1])
        rest = np.delete(w["block_tables"][b], e)  # every query is past the hole
        ref = attn.paged_attention(w["q"][q0:q1], kd, vd, rest[None], np.array([0, q1 - q0]),
                                   np.array([0, lens_q[b] + prefix[b] - 32]), w["softmax_scale"])
        err = np.abs(got[q0:q1] - ref)
        assert (err <= TOL + TOL * np.abs(ref)).all(), (b, err.max())


def test_prefill_fewer_keys_than_queries(hv, attn, cuda):  # noqa: F811
    """Lk < Lq: the first Lq - Lk queries see no key and give zeros, the others the
    causal result; a sequence without keys gives zeros."""
    lens_q, lens_k = [200, 150, 90], [130, 150, 0]
    w = _ragged(hv, [130, 150, 1], [130, 150, 1], 32, 256, 4)
    g = np.random.default_rng(1)
    q = g.standard_normal((sum(lens_q), 32, 128)).astype(np.float32)
    q = _bf16(q, "cpu").float().numpy()
    cu_q = np.concatenate([[0], np.cumsum(lens_q)]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum(lens_k)]).astype(np.int32)
    kc, vc = _bf16(w["k_cache"], cuda), _bf16(w["v_cache"], cuda)
    out = torch.full((sum(lens_q), 32, 128), float("nan"), dtype=torch.bfloat16, device=cuda)
    hv.ops.verify_attention(_bf16(q, cuda), kc, vc, torch.from_numpy(w["block_tables"]).to(cuda),
                            torch.from_numpy(cu_q).to(cuda), torch.from_numpy(cu_k).to(cuda), 200,
                            200, 128 ** -0.5, out=out)
    got = out.float().cpu().numpy()
    assert (got[:70] == 0).all() and (got[350:] == 0).all()
    for b, (q0, n) in enumerate([(70, 130), (200, 150)]):
        ref = attn.paged_attention(q[q0:q0 + n], w["k_cache"], w["v_cache"],
                                   w["block_tables"][b:b + 1], np.array([0, n]), np.array([0, n]),
                                   128 ** -0.5)
        err = np.abs(got[q0:q0 + n] - ref)
        assert (err <= TOL + TOL * np.abs(ref)).all(), (b, err.max())


def test_prefill_long_table_matches_unpaged(hv, cuda):
    """One prompt over a table of more than 64 entries, a workgroup per tile walking all
    of it, and the same rows unpaged: the same bits."""
    n = 2200
    g = torch.Generator(device=cuda).manual_seed(6)
    q = torch.randn((n, 32, 128), generator=g, device=cuda).bfloat16()
    k = torch.randn((n, 8, 128), generator=g, device=cuda).bfloat16()
    v = torch.randn((n, 8, 128), generator=g, device=cuda).bfloat16()
    cu = torch.tensor([0, n], dtype=torch.int32, device=cuda)
    nblk = -(-n // 32)
    perm = torch.randperm(nblk, generator=g, device=cuda)
    kc = torch.zeros((nblk, 32, 8, 128), dtype=torch.bfloat16, device=cuda)
    vc = torch.zeros_like(kc)
    for c, x in ((kc, k), (vc, v)):
        rows = torch.zeros((nblk * 32, 8, 128), dtype=torch.bfloat16, device=cuda)
        rows[:n] = x
        c[perm] = rows.view(nblk, 32, 8, 128)
    bt = perm.to(torch.int32)[None].contiguous()
    a = hv.ops.verify_attention(q, k, v, None, cu, cu, n, n, 128 ** -0.5)
    b = hv.ops.verify_attention(q, kc, vc, bt, cu, cu, n, n, 128 ** -0.5)
    assert torch.equal(a, b)


@pytest.mark.parametrize("kv,paged", [("bf16", True), ("fp8", True), ("bf16", False)])
def test_prefill_keeps_later_nonfinite_values_out(hv, cuda, kv, paged):
    """An infinity or NaN in a V row reaches the queries that see its key and no others:
    those before it get the same bits as without it."""
    lens = [200, 333, 150]
    g = torch.Generator(device=cuda).manual_seed(8)
    n = sum(lens)
    q = torch.randn((n, 32, 128), generator=g, device=cuda).bfloat16()
    k = torch.randn((n, 8, 128), generator=g, device=cuda).bfloat16()
    v = torch.randn((n, 8, 128), generator=g, device=cuda).bfloat16()
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device=cuda)
    dt = torch.float8_e4m3fn if kv == "fp8" else torch.bfloat16
    # (sequence, token, kv head, dim, value), one in the first, a middle and the last step
    marks = [(0, 199, 0, 5, float("nan")), (1, 31, 3, 127, float("inf")),
             (1, 97, 3, 64, float("-inf")), (2, 64, 7, 0, float("inf"))]

    def call(mark):
        vv = v.clone()
        for b, t, h, d, x in marks if mark else ():
            vv[int(cu[b]) + t, h, d] = float("nan") if kv == "fp8" else x
        if not paged:
            return hv.ops.verify_attention(q, k, vv, None, cu, cu, 333, 333, 128 ** -0.5)
        kc = torch.zeros((3, 512, 8, 128), dtype=dt, device=cuda)
        vc = torch.zeros_like(kc)
        for b, m in enumerate(lens):
            kc[b, :m] = k[int(cu[b]):int(cu[b]) + m].to(dt)
            vc[b, :m] = vv[int(cu[b]):int(cu[b]) + m].to(dt)
        bt = torch.arange(3, dtype=torch.int32, device=cuda)[:, None].contiguous()
        return hv.ops.verify_attention(q, kc, vc, bt, cu, cu, 333, 333, 128 ** -0.5)

    print(f"prefill with non-finite values {kv} paged={paged}", flush=True)
    clean, got = call(False), call(True)
    want = torch.zeros(got.shape, dtype=torch.bool, device=cuda)
    for b, t, h, d, _ in marks:
        want[int(cu[b]) + t:int(cu[b + 1]), 4 * h:4 * h + 4, d] = True
    assert torch.equal(~torch.isfinite(got), want)
    assert torch.equal(torch.where(want, clean, got), clean)


@pytest.mark.parametrize("lens_q,lens_k,declared", [
    ([1500, 1, 1, 1], [1500, 8001, 7000, 6000], 100),  # a long prompt beside cut sequences
    ([448], [8000], 200),  # the prompt itself is cut
])
def test_prefill_more_queries_than_declared(hv, cuda, lens_q, lens_k, declared):
    """A prompt longer than the declared maximum: the rows within it are those of a call
    that declares them all, the others (past the maximum's last 128-row tile) are left
    alone, the merge counters are left at zero."""
    print(f"prefill, {lens_q[0]} queries declared as {declared}", flush=True)
    B, long = len(lens_q), lens_q[0]
    g = torch.Generator(device=cuda).manual_seed(12)
    nblk = [-(-k // 256) for k in lens_k]
    kc = torch.randn((sum(nblk), 256, 8, 128), generator=g, device=cuda, dtype=torch.bfloat16)
    vc = torch.randn((sum(nblk), 256, 8, 128), generator=g, device=cuda, dtype=torch.bfloat16)
    bt = torch.full((B, max(nblk)), -1, dtype=torch.int32)
    for b, n in enumerate(nblk):
        bt[b, :n] = torch.arange(n) + sum(nblk[:b])
    bt = bt.to(cuda)
    q = torch.randn((sum(lens_q), 32, 128), generator=g, device=cuda, dtype=torch.bfloat16)
    cu_q, cu_k = (torch.tensor([sum(x[:i]) for i in range(B + 1)], dtype=torch.int32, device=cuda)
                  for x in (lens_q, lens_k))

    def call(max_q, out=None):
        return hv.ops.verify_attention(q, kc, vc, bt, cu_q, cu_k, max_q, 8192, 128 ** -0.5,
                                       out=out)

    want = call(long)
    out = torch.full_like(want, float("nan"))
    got = call(declared, out)
    ws = hv.ops.workspace(cuda, 1, "attention")
    assert int(ws[:16384].view(torch.int32).abs().max()) == 0
    written = ~torch.isnan(got).any(-1).any(-1)
    assert bool(written[:declared].all()) and bool(written[long:].all())
    assert not bool(written[-(-declared // 32) * 32:long].any())
    diff = (got[written].float() - want[written].float()).abs()
    assert float(diff.max()) <= 2e-2 * max(1.0, float(want.float().abs().max()))
    assert torch.equal(call(long), want)
