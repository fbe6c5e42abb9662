"""The pair-formulation backward at the edges of its blocks: 16-row tiles, j blocks of 24 / 16 rows, query and key
blocks of 64 / 48, the three sizes of a unit, and molecules whose units sum over several block triples, without a bias
and with bf16 and fp32 bias terms; and with values that leave fp16, or are not finite.

Bars, normwise per gradient against float64 autograd on the same rounded inputs.  bf16 gradients: the rounding of
the result (2^-9 at most, 1.7e-3 over random mantissas) with the fp16 rounding of W, dS and P (2^-11 each, random
signs under sums) below it: 4e-3.  fp32 bias gradients: they sum fp32 dS, whose error is that of S (W rounded to
fp16: 2^-11 of |S| < 4, so P is off by 2e-3 of itself at most, 6e-4 over random roundings): 2e-3.
"""

import pytest
import torch

from matterformer_amd.hip_simplicial_attention import (
    hip_simplicial_attention_backward,
    hip_simplicial_attention_forward,
)
from matterformer_amd.workloads import random_simplicial
from test_gpu_simplicial_bwd import GRAD_NAMES, abi_bwd, fp64_grads, hip_grads, logit_std, rel_err

pytestmark = pytest.mark.gpu

COUNTS = ([1, 2, 15], [16, 17, 24], [25, 47, 48], [49, 63, 64], [65, 80, 81], [97, 33], [146])


@pytest.mark.parametrize("bias_dtype", [None, torch.bfloat16, torch.float32], ids=["none", "bf16", "fp32"])
@pytest.mark.parametrize("counts", COUNTS, ids=lambda c: "n" + "-".join(map(str, c)))
def test_block_edges(cuda, counts, bias_dtype):
    """One head and a few molecules: the smallest units (8 j at most), with one query and key block or several."""
    B, H, N, D = len(counts), 1, max(counts) + 3, 64
    # a key hole and dropped pairs in the larger molecules; every query has valid pairs
    holes = [(b, 3) for b, n in enumerate(counts) if n > 20]
    case = random_simplicial(B, H, N, D, seed=sum(counts), counts=counts, holes=holes, pair_drop=0.1,
                             std=logit_std(D))
    q, k1, v1, k2, v2, qv, pkv, pv = case
    pv = pv | (torch.arange(N) < 2)[None, None, :]
    gen = torch.Generator().manual_seed(sum(counts) + 1)
    go = torch.randn(B, H, N, D, generator=gen).to(torch.bfloat16)
    ops = [t.to(torch.bfloat16) for t in (q, k1, v1, k2, v2)]
    bias = None
    if bias_dtype is not None:
        bias = [(torch.randn(B, H, N, N, generator=gen) * 0.5).to(bias_dtype) for _ in range(3)] + \
               [torch.rand(B, H, N, generator=gen).to(bias_dtype)]
    _, got = hip_grads([t.to(cuda) for t in ops], qv.to(cuda), pkv.to(cuda), pv.to(cuda), go.to(cuda), "bf16_tc",
                       bias=None if bias is None else [t.to(cuda) for t in bias])
    _, ref = fp64_grads(ops, qv, pkv, pv, go, bias=bias)
    for name, g, r in zip(GRAD_NAMES, got, ref):
        bar = 2e-3 if g.dtype == torch.float32 else 4e-3
        assert rel_err(g.float().cpu().numpy(), r) <= bar, (name, rel_err(g.float().cpu().numpy(), r))
        assert torch.isfinite(g).all(), name


def _plan(counts, heads, bias_dtype, device):
    """(units, j per unit) of the plan that mf_simplicial_bwd leaves at the start of its workspace."""
    B, N = len(counts), max(counts)
    valid = torch.arange(N)[None, :] < torch.tensor(counts)[:, None]
    ops = [torch.zeros(B, heads, N, 64, device=device, dtype=torch.bfloat16) for _ in range(5)]
    bias = None
    if bias_dtype is not None:
        bias = [torch.zeros(s, device=device, dtype=bias_dtype) for s in [(B, heads, N, N)] * 3 + [(B, heads, N)]]
    out32, lse = torch.zeros(B, heads, N, 64, device=device), torch.zeros(B, heads, N, device=device)
    *_, ws = abi_bwd(ops, ops[0], out32, lse, valid.to(device), valid.to(device), torch.float32, bias=bias)
    units, j = ws[:8].view(torch.int32).tolist()
    return units, j


@pytest.mark.parametrize("counts,bias_dtype,j,checked", [
    ([200] + [23, 24, 25, 40] * 16, None, 24, (0, 1, 2, 3, 4)),
    ([180] + [15, 16, 17, 33] * 16, torch.bfloat16, 16, (0, 1, 2, 3, 4)),
    ([180] + [15, 16, 17, 33] * 16, torch.float32, 16, (0, 1, 2, 3, 4)),
    ([128] * 16, None, 12, (7,)),
    ([64], torch.float32, 8, (0,)), ([64], torch.bfloat16, 8, (0,)),
], ids=["none-24", "bf16-16", "fp32-16", "none-12", "fp32-8", "bf16-8"])
def test_units_of_every_size(cuda, counts, bias_dtype, j, checked):
    """8 heads and enough molecules for units of 24 and 12 j (16 and 8 with a bias), whole and partial j blocks, beside
    one molecule of 200 / 180 atoms whose few units walk several j blocks of several query and key blocks (their sums
    in the slabs continue from one j block to the next).  The plan's j per unit is part of the test.  Float64 on the
    first two heads of some molecules."""
    H, D, B, N = 8, 64, len(counts), max(counts)
    assert _plan(counts, H, bias_dtype, cuda)[1] == j
    q, k1, v1, k2, v2, qv, pkv, _ = random_simplicial(B, H, N, D, seed=N, counts=counts, std=logit_std(D))
    gen = torch.Generator().manual_seed(N + 1)
    go = torch.randn(B, H, N, D, generator=gen).to(torch.bfloat16)
    ops = [t.to(torch.bfloat16) for t in (q, k1, v1, k2, v2)]
    bias = None
    if bias_dtype is not None:
        bias = [(torch.randn(B, H, N, N, generator=gen) * 0.5).to(bias_dtype) for _ in range(3)] + \
               [torch.rand(B, H, N, generator=gen).to(bias_dtype)]
    _, got = hip_grads([t.to(cuda) for t in ops], qv.to(cuda), pkv.to(cuda), None, go.to(cuda), "bf16_tc",
                       bias=None if bias is None else [t.to(cuda) for t in bias])
    for b in checked:
        n = counts[b]
        cut = lambda t: t[b:b + 1, :2, :n]  # noqa: E731
        ones = torch.ones(1, n, dtype=torch.bool)
        cbias = None if bias is None else [cut(t)[..., :n] for t in bias[:3]] + [cut(bias[3])]
        _, ref = fp64_grads([cut(t) for t in ops], ones, ones, None, cut(go), bias=cbias)
        for name, g, r in zip(GRAD_NAMES, got, ref):
            g = cut(g)[..., :n] if name in ("du", "dv_bias", "dw") else cut(g)
            bar = 2e-3 if g.dtype == torch.float32 else 4e-3
            assert rel_err(g.float().cpu().numpy(), r) <= bar, (b, n, name, rel_err(g.float().cpu().numpy(), r))


@pytest.mark.parametrize("factor", [2.0 ** -16, 2.0 ** -40, 0.0], ids=["2^-16", "2^-40", "zero"])
@pytest.mark.parametrize("bias_dtype", [None, torch.float32], ids=["none", "fp32"])
@pytest.mark.parametrize("n", [48, 100])
def test_value_rows_of_one_block_far_below_the_others(cuda, n, bias_dtype, factor):
    """The first 24 rows of v1 (or of v2) `factor` times the others: go . out, which sums over every key, is then far
    larger than any dP of a block that holds only such rows, and dS there is -P go . out.  Logits of std 5.7 let some
    of those pairs weigh in.  Bar: W rounded to fp16 moves a logit by 2^-11 of itself, |S| up to 17 (3 std) with
    random signs over d (1 / sqrt(3) and less): P off by 3e-3 where it is largest, beside the 1.7e-3 of the results'
    rounding: 6e-3, the small rows' key gradients by themselves too."""
    B, H, N, D = 1, 2, n, 64
    q, k1, v1, k2, v2, qv, pkv, _ = random_simplicial(B, H, N, D, seed=n, counts=[n], std=logit_std(D))
    q = q * 2.85
    gen = torch.Generator().manual_seed(n + 1)
    go = torch.randn(B, H, N, D, generator=gen).to(torch.bfloat16)
    bias = None
    if bias_dtype is not None:
        bias = [torch.randn(B, H, N, N, generator=gen) * 0.5 for _ in range(3)] + [torch.rand(B, H, N, generator=gen)]
    for small in (1, 2):
        w1, w2 = v1.clone(), v2.clone()
        (w1 if small == 1 else w2)[:, :, :24] *= factor
        ops = [t.to(torch.bfloat16) for t in (q, k1, w1, k2, w2)]
        _, got = hip_grads([t.to(cuda) for t in ops], qv.to(cuda), pkv.to(cuda), None, go.to(cuda), "bf16_tc",
                           bias=None if bias is None else [t.to(cuda) for t in bias])
        _, ref = fp64_grads(ops, qv, pkv, None, go, bias=bias)
        for name, g, r in zip(GRAD_NAMES, got, ref):
            g = g.float().cpu().numpy()
            assert rel_err(g, r) <= 6e-3, (small, name, rel_err(g, r))
            if name == f"dk{small}":
                e = rel_err(g[:, :, :24], r[:, :, :24])
                assert e <= 6e-3, (small, name, "small rows", e)


@pytest.mark.parametrize("n", [128, 384, 512])
def test_flat_softmax_of_a_large_molecule(cuda, n):
    """Logits of std 0.2 over n^2 pairs: every P is near n^-2 (2^-18 at 512 tokens), below fp16's normal range unless
    it is scaled, and only rounding to nearest averages out in dv1 and dv2 (unscaled and truncated: 8.7e-3).  Bar:
    the bf16 result's 1.7e-3 with the fp16 roundings of W, P and dS (2.8e-4 rms each) below it: 2.2e-3.  The float64
    reference runs on the GPU."""
    H, D = 1, 64
    q, k1, v1, k2, v2, *_ = random_simplicial(1, H, n, D, seed=n, counts=[n], std=logit_std(D))
    go = torch.randn(1, H, n, D, generator=torch.Generator().manual_seed(n)).to(torch.bfloat16).to(cuda)
    ops = [t.to(torch.bfloat16).to(cuda) for t in (q * 0.1, k1, v1, k2, v2)]
    valid = torch.ones(1, n, dtype=torch.bool, device=cuda)
    _, got = hip_grads(ops, valid, valid, None, go, "bf16_tc")
    leaves = [t[0].double().requires_grad_(True) for t in ops]
    a, b, c, d, e = leaves
    logits = torch.matmul((a[:, :, None] * b[:, None]).reshape(H, n * n, D), d.transpose(1, 2).contiguous())
    p = torch.softmax(logits.view(H, n, n * n), dim=-1).view(H, n * n, n)
    out = (torch.matmul(p, e).view(H, n, n, D) * c[:, None]).sum(2)
    for name, g, r in zip(GRAD_NAMES, got, torch.autograd.grad(out, leaves, go[0].double())):
        assert rel_err(g[0].float().cpu().numpy(), r.cpu().numpy()) <= 2.2e-3, name


@pytest.mark.parametrize("value", [float("nan"), float("inf")], ids=["nan", "inf"])
@pytest.mark.parametrize("which", ["q", "go"])
@pytest.mark.parametrize("n", [20, 90, 150])
def test_a_row_that_is_not_finite_leaves_the_other_queries_alone(cuda, n, which, value):
    """NaN or infinity in one row of q or grad_out: dq, du, dv_bias and dgate of the other queries are those of the
    call without it (the sums over queries are NaN, as they should be)."""
    B, H, D, bad = 1, 2, 64, 3
    q, k1, v1, k2, v2, qv, pkv, _ = random_simplicial(B, H, n, D, seed=n, counts=[n], std=logit_std(D))
    gen = torch.Generator().manual_seed(n)
    go = torch.randn(B, H, n, D, generator=gen).to(torch.bfloat16)
    ops = [t.to(torch.bfloat16) for t in (q, k1, v1, k2, v2)]
    for bias in (None, [torch.randn(B, H, n, n, generator=gen) * 0.5 for _ in range(3)] +
                 [torch.rand(B, H, n, generator=gen)]):
        _, ref = fp64_grads(ops, qv, pkv, None, go, bias=bias)
        x = [t.clone() for t in (*ops, go)]
        x[0 if which == "q" else 5][:, :, bad, 7] = value
        _, got = hip_grads([t.to(cuda) for t in x[:5]], qv.to(cuda), pkv.to(cuda), None, x[5].to(cuda), "bf16_tc",
                           bias=None if bias is None else [t.to(cuda) for t in bias])
        others = [i for i in range(n) if i != bad]
        for name, g, r in zip(GRAD_NAMES, got, ref):
            if name in ("dq", "du", "dv_bias", "dgate") and g is not None:
                bar = 2e-3 if g.dtype == torch.float32 else 4e-3
                e = rel_err(g.float().cpu().numpy()[:, :, others], r[:, :, others])
                assert e <= bar, (name, e)


def test_lse_far_too_small_gives_large_gradients_not_nan(cuda):
    """A forward that saturated its bias terms returns an lse below the backward's own logits: P up to e^10 leaves
    fp16, where it becomes the largest fp16."""
    n = 40
    q, k1, v1, k2, v2, *_ = random_simplicial(1, 2, n, 64, seed=1, counts=[n], std=logit_std(64))
    ops = [t.to(torch.bfloat16).to(cuda) for t in (q, k1, v1, k2, v2)]
    masks = dict.fromkeys(("query_valid", "pair_key_valid"), torch.ones(1, n, dtype=torch.bool, device=cuda))
    masks["pair_valid"] = None
    _, lse, out32 = hip_simplicial_attention_forward(*ops, **masks)
    for g in hip_simplicial_attention_backward(ops[0], *ops, out32, lse - 10.0, **masks)[:5]:
        assert torch.isfinite(g).all()


def test_gradients_below_the_fp32_range_are_zero_not_nan(cuda):
    """go of 1e-6 and v1 of 2^-110: dS is below 2^-126, so dq, dk1 and dk2 vanish; dv1 does not.  (2^-es of such a
    block, unbounded, is infinite, and infinity times the zeros of dropped pairs was NaN.)"""
    B, H, N, D = 1, 2, 48, 64
    q, k1, v1, k2, v2, qv, pkv, pv = random_simplicial(B, H, N, D, seed=9, counts=[48], pair_drop=0.2, std=logit_std(D))
    pv = pv | (torch.arange(N) < 2)[None, None, :]
    go = torch.randn(B, H, N, D, generator=torch.Generator().manual_seed(10)) * 1e-6
    ops = [t.to(torch.bfloat16) for t in (q, k1, v1 * 2.0 ** -110, k2, v2)]
    go = go.to(torch.bfloat16)
    _, got = hip_grads([t.to(cuda) for t in ops], qv.to(cuda), pkv.to(cuda), pv.to(cuda), go.to(cuda), "bf16_tc")
    _, ref = fp64_grads(ops, qv, pkv, pv, go)
    for name, g, r in zip(GRAD_NAMES, got, ref):
        g = g.float().cpu()
        assert torch.isfinite(g).all(), name
        if name in ("dq", "dk1", "dk2", "dv2"):
            assert float(g.abs().max()) <= 2.0 ** -110, name
        else:
            assert rel_err(g.numpy(), r) <= 4e-3, (name, rel_err(g.numpy(), r))


@pytest.mark.parametrize("counts,heads,bias_dtype,want", [
    ([72] * 16, 8, None, (384, 24)),               # one round; not 768 units of 12 rows
    ([64], 8, torch.float32, (64, 8)),             # half the parts to add for the same round
    ([192] * 4, 12, torch.bfloat16, (576, 16)),    # 64 units left for the second round, not 1152 of 8 rows
    ([64] * 256, 8, None, (6144, 24)),             # many rounds: fewer, longer units
    ([256], 8, None, (256, 6)),                    # whole rounds of four key pairs: 8 rows
    ([128] * 16, 8, None, (1024, 12)), ([44] * 64, 8, None, (1024, 24)), ([44, 9, 30], 2, None, (24, 6)),
], ids=lambda v: str(v) if isinstance(v, int) else None)
def test_rows_per_unit(cuda, counts, heads, bias_dtype, want):
    """The schedule takes the j per unit whose units finish first on the chip's 512 slots."""
    assert _plan(counts, heads, bias_dtype, cuda) == want


def test_queries_and_keys_of_different_counts(cuda):
    """More queries than keys and the reverse (70 / 20 and 20 / 70 valid rows): blocks of one side only."""
    B, H, N, D = 2, 2, 75, 64
    q, k1, v1, k2, v2, qv, pkv, _ = random_simplicial(B, H, N, D, seed=5, counts=[70, 70], std=logit_std(D))
    qv, pkv = qv.clone(), pkv.clone()
    pkv[0, 20:] = False
    qv[1, 20:] = False
    gen = torch.Generator().manual_seed(6)
    go = torch.randn(B, H, N, D, generator=gen).to(torch.bfloat16)
    ops = [t.to(torch.bfloat16) for t in (q, k1, v1, k2, v2)]
    bias = [torch.randn(B, H, N, N, generator=gen) * 0.5 for _ in range(3)] + [torch.rand(B, H, N, generator=gen)]
    _, got = hip_grads([t.to(cuda) for t in ops], qv.to(cuda), pkv.to(cuda), None, go.to(cuda), "bf16_tc",
                       bias=[t.to(cuda) for t in bias])
    _, ref = fp64_grads(ops, qv, pkv, None, go, bias=bias)
    for name, g, r in zip(GRAD_NAMES, got, ref):
        bar = 2e-3 if g.dtype == torch.float32 else 4e-3
        assert rel_err(g.float().cpu().numpy(), r) <= bar, (name, rel_err(g.float().cpu().numpy(), r))


@pytest.mark.parametrize("bias_dtype", [None, torch.bfloat16, torch.float32], ids=["none", "bf16", "fp32"])
def test_without_memory_for_the_workspace(cuda, bias_dtype, monkeypatch):
    """When the workspace cannot be allocated the call runs on the ownership kernel (bf16 products, 2e-2 as in its
    own tests), with an fp32 bias after the entry that writes the leaves' dtypes has refused it."""
    import matterformer_amd.hip_simplicial_attention as hsa

    B, H, N, D = 2, 2, 70, 64
    q, k1, v1, k2, v2, qv, pkv, pv = random_simplicial(B, H, N, D, seed=11, counts=[70, 33], pair_drop=0.1,
                                                       std=logit_std(D))
    pv = pv | (torch.arange(N) < 2)[None, None, :]
    gen = torch.Generator().manual_seed(12)
    go = torch.randn(B, H, N, D, generator=gen).to(torch.bfloat16)
    ops = [t.to(torch.bfloat16) for t in (q, k1, v1, k2, v2)]
    bias = None
    if bias_dtype is not None:
        bias = [(torch.randn(B, H, N, N, generator=gen) * 0.5).to(bias_dtype) for _ in range(3)] + \
               [torch.rand(B, H, N, generator=gen).to(bias_dtype)]
    args = [[t.to(cuda) for t in ops], qv.to(cuda), pkv.to(cuda), pv.to(cuda), go.to(cuda), "bf16_tc"]
    dbias = None if bias is None else [t.to(cuda) for t in bias]
    _, usual = hip_grads(*args, bias=dbias)
    real, refused = torch.empty, []

    def empty(*a, **k):
        if k.get("dtype") == torch.uint8:
            refused.append(a)
            raise torch.OutOfMemoryError("no memory")
        return real(*a, **k)

    monkeypatch.setattr(hsa.torch, "empty", empty)
    _, got = hip_grads(*args, bias=dbias)
    monkeypatch.undo()
    assert len(refused) == (2 if bias_dtype == torch.float32 else 1)
    _, ref = fp64_grads(ops, qv, pkv, pv, go, bias=bias)
    for name, g, u, r in zip(GRAD_NAMES, got, usual, ref):
        assert g.dtype == u.dtype
        assert rel_err(g.float().cpu().numpy(), r) <= 2e-2, name
        pad = torch.from_numpy(r == 0.0).to(cuda)
        assert not g[pad].any(), name


@pytest.mark.parametrize("wanted", [(True, True, True, True), (False, True, False, False)], ids=["all", "dv"])
@pytest.mark.parametrize("B,N", [(1, 9), (3, 45), (2, 130)])
def test_gradients_in_the_leaves_dtypes_are_written_in_full(cuda, B, N, wanted):
    """bf16 operands with an fp32 bias: the entry that writes every element gives what the zero-filled fp32
    gradients cast to the leaves' dtypes give, bit for bit (the same sums, rounded once), over buffers that held
    NaN, padded rows included."""
    import matterformer_amd.hip_simplicial_attention as hsa

    H, D = 1, 64
    counts = [max(1, N - 7 * b - 4) for b in range(B)]
    q, k1, v1, k2, v2, qv, pkv, pv = random_simplicial(B, H, N, D, seed=N, counts=counts, pair_drop=0.1,
                                                       std=logit_std(D))
    gen = torch.Generator().manual_seed(N + 1)
    ops = [t.to(torch.bfloat16).to(cuda) for t in (q, k1, v1, k2, v2)]
    go = torch.randn(B, H, N, D, generator=gen).to(torch.bfloat16).to(cuda)
    bias = [(torch.randn(s, generator=gen) * 0.5).to(cuda) for s in [(B, H, N, N)] * 3 + [(B, H, N)]]
    masks = dict(query_valid=qv.to(cuda), pair_key_valid=pkv.to(cuda), pair_valid=pv.to(cuda))
    _, lse, out32 = hsa.hip_simplicial_attention_forward(*ops, **masks, u=bias[0], v_bias=bias[1], w=bias[2],
                                                         gate=bias[3])
    flags = dict.fromkeys([f"need_d{n}" for n in ("u", "v_bias", "w", "gate", "angle_left", "angle_right", "angle_gate",
                                                  "message_left", "message_right", "message_basis")], False)
    flags.update(zip(("need_du", "need_dv_bias", "need_dw", "need_dgate"), wanted))
    call = (go, *ops, out32, lse, *masks.values(), *bias, *[None] * 6, flags)
    want = hsa._kernel_backward(*call, allow_leaf=False)
    real = torch.empty
    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(hsa.torch, "empty", lambda *a, **k: real(*a, **k).fill_(float("nan"))
                   if k.get("dtype") in (torch.float32, torch.bfloat16) else real(*a, **k))
        got = hsa._kernel_backward(*call)
    for g, w in zip(got, want):
        assert (g is None) == (w is None)
        if w is not None:
            assert g.dtype == w.dtype and torch.equal(g, w)


def test_leaf_entry_refuses_other_calls():
    """grads_dtype F32 or a bias of another dtype is refused before anything is read or launched."""
    from matterformer_amd import _native

    lib = _native.lib()
    fake = 4096
    for grads, bias in ((_native.MF_DTYPE_F32, _native.MF_DTYPE_F32), (_native.MF_DTYPE_BF16, _native.MF_DTYPE_BF16)):
        a = _native.MfSimplicialBwdArgs(q=fake, k1=fake, v1=fake, k2=fake, v2=fake, grad_out=fake, out=fake, lse=fake,
                                        query_valid=fake, pair_key_valid=fake, bias_u=fake, bias_v=fake, bias_w=fake,
                                        bias_gate=fake, bias_dtype=bias, grads_dtype=grads, batch=1, heads=1,
                                        tokens=8, head_dim=64)
        assert lib.mf_simplicial_bwd_leaf(a, None) == _native.MF_ERR_INVALID_ARGUMENT
