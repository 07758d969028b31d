"""GPU parity of the listed attention launches (batches of more sequences than the
static grid holds at once): the splits come from the real lengths, so short,
long, empty-handed and one-key sequences share a call. Fused entry against the
two launches bit for bit, and against the float64 oracle within 2e-2."""
import numpy as np
import pytest
import torch

from test_gpu_fused_ops import _attend_inputs, _norm_rope_ref, _rope_table

pytestmark = pytest.mark.gpu

# (name, Hq, Hkv, query lengths, earlier keys, block size, declared max_seqlen_k):
# pairs of a length at a split's or window's edge; 64 sequences, the most; one long
# sequence among short ones (many splits of one); sequences past 4096 keys; past 8192
# (the longest split); more splits asked for than the partials' share of the workspace
# holds; 4 and 16 kv heads (other CUs per head); G = 1 with 16 query rows, and 8
_CASES = [
    ("edges", 32, 8, [4] * 12, [0, 28, 60, 508, 509, 1020, 1021, 1531, 1, 33, 700, 2044], 256,
     4101),
    ("most", 16, 8, [1, 2, 3, 4] * 16, [(37 * i) % 900 for i in range(64)], 32, 4101),
    ("one-long", 32, 8, [4] * 16, [4000] + [3 * i for i in range(15)], 256, 4101),
    ("past-4096", 16, 8, [2] * 17, [6000, 4094, 4095] + [200 * i for i in range(14)], 256, 8200),
    ("past-8192", 16, 8, [2] * 10, [12000, 8190, 8191, 9000, 5, 300, 0, 64, 8192, 2000], 256,
     12300),
    ("partials", 16, 8, [1] * 64, [4200] + [29 * i for i in range(63)], 256, 4220),
    ("group-8", 64, 8, [2, 1] * 8, [2000, 0, 31, 700] * 4, 256, 4101),
    ("heads-4", 16, 4, [4] * 33, [50 * i for i in range(33)], 64, 4101),
    ("heads-16", 16, 16, [16] * 9, [31, 300, 0, 77, 500, 1000, 5, 16, 90], 96, 2100),
]


@pytest.mark.parametrize("kv", ["bf16", "fp8"])
@pytest.mark.parametrize("case", _CASES, ids=[c[0] for c in _CASES])
def test_listed_attention(hv, cuda, kv, case):
    from oracle import attn as oa
    ops = hv.ops
    x = _attend_inputs(cuda, kv, case)
    x["cs"] = _rope_table(12400, cuda)  # every position of the cases
    Hq, Hkv = x["Hq"], x["Hkv"]
    print(f"listed attention {case[0]} kv={kv} B={x['B']}", flush=True)
    kc1, vc1, kc2, vc2 = x["kc"], x["vc"], x["kc"].clone(), x["vc"].clone()
    scales = dict(k_scale=x["ksc"], v_scale=x["vsc"])
    norm = (x["qkv"], Hq, Hkv, x["qw"], x["kw"], x["cs"], x["pos"], 1e-6)
    # two calls each: the split tickets are left at zero
    for _ in range(2):
        q = ops.qk_norm_rope_store(*norm, kc1, vc1, x["slots"], **scales)
        out1 = ops.verify_attention(q, kc1, vc1, x["bt"], x["cu_q"], x["cu_k"], x["max_q"],
                                    x["max_k"], 128 ** -0.5, **scales)
        out2 = ops.qk_norm_rope_attend(*norm, kc2, vc2, x["slots"], x["bt"], x["cu_q"],
                                       x["cu_k"], x["max_q"], x["max_k"], 128 ** -0.5, **scales)
        assert torch.equal(out1.view(torch.int16), out2.view(torch.int16))
    assert torch.equal(kc1.view(torch.uint8), kc2.view(torch.uint8))
    assert torch.equal(vc1.view(torch.uint8), vc2.view(torch.uint8))
    if kv == "bf16":
        kd, vd = kc2.float().cpu().numpy(), vc2.float().cpu().numpy()
    else:
        kd = oa.dequant(kc2.view(torch.uint8).cpu().numpy(), x["ksc"])
        vd = oa.dequant(vc2.view(torch.uint8).cpu().numpy(), x["vsc"])
    qr = _norm_rope_ref(x["qkv"].cpu()[:, :Hq * 128].view(-1, Hq, 128), x["qw"].cpu(),
                        x["cs"].cpu(), x["pos"].cpu(), 1e-6)
    ref = oa.paged_attention(qr.float().numpy(), kd, vd, x["bt"].cpu().numpy(),
                             x["cu_q"].cpu().numpy(), x["cu_k"].cpu().numpy(), 128 ** -0.5)
    err = np.abs(out2.float().cpu().numpy() - ref).max()
    assert err <= 2e-2 * max(1.0, np.abs(ref).max()), err


def test_listed_keys_past_the_declared_maximum(hv, cuda):
    """Sequences longer than the declared maximum: the list holds no more entries than the
    launch has workgroups, so every row is written and the merge counters are left at
    zero, and the next call in the same workspace is right."""
    B, Hq, Hkv, declared, keys = 48, 16, 8, 2048, 9000
    print("listed attention, 48 sequences of 9000 keys declared as 2048", flush=True)
    g = torch.Generator(device=cuda).manual_seed(11)
    nblk = -(-keys // 256)
    kc = torch.randn((B * nblk, 256, Hkv, 128), generator=g, device=cuda, dtype=torch.bfloat16)
    vc = torch.randn((B * nblk, 256, Hkv, 128), generator=g, device=cuda, dtype=torch.bfloat16)
    bt = torch.arange(B * nblk, dtype=torch.int32, device=cuda).view(B, nblk)
    q = torch.randn((B, Hq, 128), generator=g, device=cuda, dtype=torch.bfloat16)
    cu_q = torch.arange(B + 1, dtype=torch.int32, device=cuda)

    def call(n, out=None):
        return hv.ops.verify_attention(q, kc, vc, bt, cu_q, cu_q * n, 1, declared, 128 ** -0.5,
                                       out=out)

    want = call(1500)
    out = torch.full_like(q, float("nan"))
    call(keys, out)
    assert not torch.isnan(out).any()
    ws = hv.ops.workspace(cuda, 1, "attention")
    assert int(ws[:16384].view(torch.int32).abs().max()) == 0
    assert torch.equal(call(1500), want)


def test_calls_without_splits_leave_the_workspace_alone(hv, cuda):
    """48 short sequences, more workgroups than CUs, no key split: the call neither reads
    nor writes its workspace (calls of this kind may overlap on two streams)."""
    lens = [40 + 12 * i for i in range(48)]
    x = _attend_inputs(cuda, "bf16", ("short", 16, 8, [4] * 48, [n - 4 for n in lens], 256, 640))
    print("attention without splits, 48 sequences of up to 604 keys", flush=True)
    norm = (x["qkv"], 16, 8, x["qw"], x["kw"], x["cs"], x["pos"], 1e-6)
    tail = (x["bt"], x["cu_q"], x["cu_k"], x["max_q"], x["max_k"], 128 ** -0.5)
    need = hv._lib.lib().hs_verify_attention_workspace_size(48, 16, 8, 4, x["max_k"])
    ws = hv.ops.workspace(cuda, need, "attention")

    def both():
        q = hv.ops.qk_norm_rope_store(*norm, x["kc"], x["vc"], x["slots"])
        return (hv.ops.verify_attention(q, x["kc"], x["vc"], *tail),
                hv.ops.qk_norm_rope_attend(*norm, x["kc"], x["vc"], x["slots"], *tail))

    want = both()
    saved = ws.clone()
    ws.fill_(0xA5)
    try:
        got = both()
        assert bool((ws == 0xA5).all())
    finally:
        ws.copy_(saved)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
