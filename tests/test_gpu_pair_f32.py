"""The fp32 pair-formulation kernels at the edges of their tiles and of the range they serve (forward at most 64
tokens and head_dim 64, backward 32 and 32; larger calls, and few molecules of 49 / 25 tokens and more without a bias,
run the general kernels), in both shapes of their workgroups, with and without a factorized bias, against float64 on
the same inputs.

Bar, normwise per result: products and sums are fp32 over at most n^2 = 4096 terms in short chains; 2^-24 per
rounding with random signs over the chains (about 20 roundings a term) gives below 1e-6, and the hardware exp2's
1 ulp of arguments up to 30 another 1e-6: 4e-6.  With offsets near 300 (log2 units) the argument itself is rounded
to 2^-24 * 300 = 2e-5 of P: 4e-5 there."""

import pytest
import torch

from matterformer_amd.hip_simplicial_attention import hip_simplicial_attention_forward
from matterformer_amd.workloads import random_simplicial
from test_gpu_simplicial_bwd import GRAD_NAMES, fp64_grads, hip_grads, logit_std, rel_err

pytestmark = pytest.mark.gpu

SHAPES = [([1, 2, 15], 4), ([16, 17, 9], 32), ([31, 32, 5], 32), ([29, 32], 20), ([32, 16], 64), ([33, 48], 32),
          ([49, 64], 36), ([65, 12], 32)]


@pytest.mark.parametrize("bias_dtype", [None, torch.float32, torch.bfloat16], ids=["none", "fp32", "bf16"])
@pytest.mark.parametrize("counts,D", SHAPES, ids=lambda v: "-".join(map(str, v)) if isinstance(v, list) else f"D{v}")
def test_fp32_tile_edges(cuda, counts, D, bias_dtype):
    B, H, N = len(counts), 2, max(counts)
    holes = [(b, 2) for b, n in enumerate(counts) if n > 8]
    q, k1, v1, k2, v2, qv, pkv, pv = random_simplicial(B, H, N, D, seed=N + D, counts=counts, holes=holes,
                                                       pair_drop=0.1, std=logit_std(D))
    pv = pv | (torch.arange(N) < 2)[None, None, :]  # every query has valid pairs
    gen = torch.Generator().manual_seed(N * 3 + D)
    go = torch.randn(B, H, N, D, generator=gen)
    bias = None
    if bias_dtype is not None:
        bias = [(torch.randn(B, H, N, N, generator=gen) * 0.5).to(bias_dtype) for _ in range(3)] + \
               [torch.randn(B, H, N, generator=gen).to(bias_dtype)]
    ops = [q, k1, v1, k2, v2]
    out, got = hip_grads([t.to(cuda) for t in ops], qv.to(cuda), pkv.to(cuda), pv.to(cuda), go.to(cuda), "ieee_fp32",
                         bias=None if bias is None else [t.to(cuda) for t in bias])
    want, ref = fp64_grads(ops, qv, pkv, pv, go, bias=bias)
    assert rel_err(out.cpu().numpy(), want) <= 4e-6
    for name, g, r in zip(GRAD_NAMES, got, ref):
        # a bf16 bias gets bf16 gradients (rounding 2^-9, 1.7e-3 normwise)
        bar = 4e-3 if g.dtype == torch.bfloat16 else 4e-6
        assert rel_err(g.float().cpu().numpy(), r) <= bar, name


@pytest.mark.parametrize("n,D,bar", [(29, 32, 7.5e-7), (29, 64, 1.05e-6), (48, 64, 1.1e-6)])
def test_backward_sums_the_logits_as_the_forward_does(cuda, n, D, bar):
    """Gradients of calls whose forward runs in pair form, over 8 molecules of 4 heads.  The matrix cores' fp32 sums
    err to one side along a chain, so lse and the backward's S have to sum in chains of the same length: with S in
    one chain of D / 4 steps and the forward's lse from two, the errors were 9.5e-7 .. 1.1e-6 (29 tokens, head_dim
    32), 1.1e-6 .. 1.25e-6 (head_dim 64) and 1.2e-6 .. 1.4e-6 (48, 64).  The rounding of lse (8 .. 9, 2.8e-7 rms), of
    lse log2 e and of exp2's argument (2e-7 each) make 4e-7, which adds to the chains' 4e-7 at D = 32 and 8e-7 at 64."""
    B, H = 8, 4
    q, k1, v1, k2, v2, qv, pkv, _ = random_simplicial(B, H, n, D, seed=n + D, counts=[n] * B, std=logit_std(D))
    go = torch.randn(B, H, n, D, generator=torch.Generator().manual_seed(D))
    ops = [q, k1, v1, k2, v2]
    _, got = hip_grads([t.to(cuda) for t in ops], qv.to(cuda), pkv.to(cuda), None, go.to(cuda), "ieee_fp32")
    _, ref = fp64_grads(ops, qv, pkv, None, go)
    for name, g, r in zip(GRAD_NAMES, got, ref):
        assert rel_err(g.cpu().numpy(), r) <= bar, (name, rel_err(g.cpu().numpy(), r))


@pytest.mark.parametrize("with_bias", [False, True], ids=["none", "bias"])
@pytest.mark.parametrize("B,H,n,D", [(32, 8, 16, 32), (33, 8, 16, 32), (16, 8, 31, 32), (17, 8, 32, 32), (40, 4, 33, 64),
                                     (8, 8, 64, 64), (9, 8, 64, 20), (4, 8, 64, 32), (4, 8, 49, 64), (5, 8, 49, 32)])
def test_both_workgroup_shapes_of_the_forward(cuda, B, H, n, D, with_bias):
    """Calls on either side of the line between one query tile a workgroup of eight waves (one workgroup per CU at
    most) and two tiles of four waves, and of the line past which few molecules of 49 tokens and more take the general
    kernel (without a bias, 32 (molecule, head)): the same outputs as the molecules one by one, and as float64."""
    counts = [n - b % 3 for b in range(B)]
    q, k1, v1, k2, v2, qv, pkv, _ = random_simplicial(B, H, n, D, seed=B + n, counts=counts, std=logit_std(D))
    gen = torch.Generator().manual_seed(B)
    bias = None
    if with_bias:
        bias = [torch.randn(B, H, n, n, generator=gen) * 0.5 for _ in range(3)] + [torch.rand(B, H, n, generator=gen)]
    ops = [t.to(cuda) for t in (q, k1, v1, k2, v2)]
    masks = [qv.to(cuda), pkv.to(cuda)]

    def forward(s):
        kw = {} if bias is None else {k: t[s].to(cuda) for k, t in zip(("u", "v_bias", "w", "gate"), bias)}
        return hip_simplicial_attention_forward(*[t[s] for t in ops], query_valid=masks[0][s], pair_key_valid=masks[1][s],
                                                pair_valid=None, precision="ieee_fp32", **kw)

    out, lse, _ = forward(slice(0, B))
    for b in (0, B - 1):
        s = slice(b, b + 1)
        o1, l1, _ = forward(s)
        assert rel_err(out[s].cpu().numpy(), o1.cpu().double().numpy()) <= 4e-6
        assert rel_err(lse[s].cpu().numpy(), l1.cpu().double().numpy()) <= 4e-6
        zero = torch.zeros(1, H, n, D)
        want, _ = fp64_grads([t[s] for t in (q, k1, v1, k2, v2)], qv[s], pkv[s], None, zero,
                             bias=None if bias is None else [t[s] for t in bias])
        assert rel_err(out[s].cpu().numpy(), want) <= 4e-6


@pytest.mark.parametrize("with_bias", [False, True], ids=["none", "bias"])
@pytest.mark.parametrize("B,n,D", [(64, 17, 32), (65, 17, 32), (65, 32, 20), (66, 9, 32)])
def test_both_workgroup_shapes_of_the_backward(cuda, B, n, D, with_bias):
    """Eight waves a (molecule, head) up to one workgroup per CU (256), four past it; bar as above."""
    H = 4
    counts = [n - b % 4 for b in range(B)]
    q, k1, v1, k2, v2, qv, pkv, _ = random_simplicial(B, H, n, D, seed=B + n, counts=counts, std=logit_std(D))
    gen = torch.Generator().manual_seed(B)
    go = torch.randn(B, H, n, D, generator=gen)
    bias = None
    if with_bias:
        bias = [torch.randn(B, H, n, n, generator=gen) * 0.5 for _ in range(3)] + [torch.rand(B, H, n, generator=gen)]
    ops = [q, k1, v1, k2, v2]
    _, got = hip_grads([t.to(cuda) for t in ops], qv.to(cuda), pkv.to(cuda), None, go.to(cuda), "ieee_fp32",
                       bias=None if bias is None else [t.to(cuda) for t in bias])
    _, ref = fp64_grads(ops, qv, pkv, None, go, bias=bias)
    for name, g, r in zip(GRAD_NAMES, got, ref):
        assert rel_err(g.cpu().numpy(), r) <= 4e-6, name


def test_large_and_masking_scale_logits(cuda):
    """Logits far past the first tile's maximum in both directions (the offset moves many times) and bias terms of
    -30000 beside ordinary ones; padded queries, a molecule without keys and one without queries give zeros."""
    B, H, N, D = 4, 2, 29, 32
    q, k1, v1, k2, v2, qv, pkv, _ = random_simplicial(B, H, N, D, seed=3, counts=[29, 20, 9, 9], std=logit_std(D))
    q = q * 60.0
    qv, pkv = qv.clone(), pkv.clone()
    pkv[2] = False
    qv[3] = False
    gen = torch.Generator().manual_seed(4)
    u, v, w = (torch.randn(B, H, N, N, generator=gen) for _ in range(3))
    w[torch.rand(B, H, N, N, generator=gen) < 0.3] = -30000.0
    bias = [u, v, w, torch.rand(B, H, N, generator=gen) + 0.5]
    ops = [q, k1, v1, k2, v2]
    kw = dict(u=bias[0], v_bias=bias[1], w=bias[2], gate=bias[3])
    out, lse, out32 = hip_simplicial_attention_forward(
        *[t.to(cuda) for t in ops], query_valid=qv.to(cuda), pair_key_valid=pkv.to(cuda), pair_valid=None,
        precision="ieee_fp32", **{k: t.to(cuda) for k, t in kw.items()})
    torch.cuda.synchronize()
    go = torch.randn(B, H, N, D, generator=gen)
    sub = slice(0, 2)
    want, _ = fp64_grads([t[sub] for t in ops], qv[sub], pkv[sub], None, go[sub], bias=[t[sub] for t in bias])
    assert rel_err(out[sub].cpu().numpy(), want) <= 4e-5
    assert torch.equal(out, out32)
    assert not out[2:].any() and not lse[2:].any()
    assert not out[1, :, 20:].any() and not lse[1, :, 20:].any()


# operands, bias, head_dim, tokens, bars of the operand and bias gradients (bf16 operands: the bars of the block tests)
INFINITE = [(torch.float32, torch.float32, 32, 20, 4e-6, 4e-6), (torch.float32, torch.float32, 64, 20, 4e-6, 4e-6),
            (torch.bfloat16, torch.bfloat16, 64, 20, 4e-3, 4e-3), (torch.bfloat16, torch.float32, 64, 20, 4e-3, 2e-3),
            (torch.bfloat16, torch.float32, 64, 90, 4e-3, 2e-3)]


@pytest.mark.parametrize("dtype,bias_dtype,D,n,bar,bias_bar", INFINITE,
                         ids=lambda v: str(v).replace("torch.", "") if not isinstance(v, float) else None)
@pytest.mark.parametrize("term", ["-inf dropped", "nan dropped", "-inf kept"])
def test_bias_terms_that_are_not_finite(cuda, dtype, bias_dtype, D, n, bar, bias_bar, term):
    """-inf or NaN terms at pairs that pair_valid drops count for nothing; -inf at pairs that it keeps is a mask of
    its own (P = 0 for every query), and every gradient but dgate, whose sum has 0 * -inf, is finite.  20 and 90
    tokens leave padding rows in the last query tile."""
    B, H = 1, 2
    q, k1, v1, k2, v2, qv, pkv, _ = random_simplicial(B, H, n, D, seed=n + D, counts=[n], std=logit_std(D))
    gen = torch.Generator().manual_seed(n)
    pv = torch.rand(B, n, n, generator=gen) < 0.8
    pv[:, :, :2] = True
    go = torch.randn(B, H, n, D, generator=gen).to(dtype)
    ops = [t.to(dtype) for t in (q, k1, v1, k2, v2)]
    bias = [(torch.randn(B, H, n, n, generator=gen) * 0.5).to(bias_dtype) for _ in range(3)] + \
           [(torch.rand(B, H, n, generator=gen) + 0.5).to(bias_dtype)]
    at = ~pv[:, None].expand(B, H, n, n)
    bias[2][at] = 0.0
    plain = [t.clone() for t in bias]
    bias[2][at] = float(term.split()[0])
    kept = term.endswith("kept")
    mask = None if kept else pv
    _, got = hip_grads([t.to(cuda) for t in ops], qv.to(cuda), pkv.to(cuda), None if kept else pv.to(cuda), go.to(cuda),
                       "ieee_fp32" if dtype == torch.float32 else "bf16_tc", bias=[t.to(cuda) for t in bias])
    _, ref = fp64_grads(ops, qv, pkv, mask, go, bias=bias if kept else plain)
    for name, g, r in zip(GRAD_NAMES, got, ref):
        if kept and name == "dgate":
            continue
        assert torch.isfinite(g).all(), name
        e = rel_err(g.float().cpu().numpy(), r)
        assert e <= (bias_bar if name in GRAD_NAMES[5:] else bar), (name, e)


@pytest.mark.parametrize("wanted", [(True, True, True, True), (False, True, False, False)], ids=["all", "dv"])
@pytest.mark.parametrize("counts,N,D", [([1, 3], 4, 4), ([16, 9, 0], 17, 20), ([32, 5], 32, 32), ([29, 12], 29, 32)])
def test_gradients_are_written_in_full(cuda, counts, N, D, wanted):
    """Over buffers that held NaN, every padded entry of the fp32 gradients is zero and the others are those of the
    same call into zero-filled buffers, bit for bit (the sums do not depend on what the buffers held); queries and
    keys padded differently, a molecule without either."""
    import matterformer_amd.hip_simplicial_attention as hsa

    B, H = len(counts), 2
    q, k1, v1, k2, v2, qv, pkv, _ = random_simplicial(B, H, N, D, seed=N, counts=counts, std=logit_std(D))
    qv = qv.clone()
    qv[0, counts[0] // 2:] = False
    if B > 1:
        qv[1, 0] = True  # a query past the keys' count too when there are no keys
    gen = torch.Generator().manual_seed(N)
    ops = [t.to(cuda) for t in (q, k1, v1, k2, v2)]
    go = torch.randn(B, H, N, D, generator=gen).to(cuda)
    bias = [torch.randn(s, generator=gen).to(cuda) for s in [(B, H, N, N)] * 3 + [(B, H, N)]]
    masks = (qv.to(cuda), pkv.to(cuda), None)
    kw = dict(zip(("query_valid", "pair_key_valid", "pair_valid"), masks))
    flags = dict.fromkeys([f"need_d{n}" for n in ("u", "v_bias", "w", "gate", "angle_left", "angle_right", "angle_gate",
                                                  "message_left", "message_right", "message_basis")], False)
    flags.update(zip(("need_du", "need_dv_bias", "need_dw", "need_dgate"), wanted))
    for b in (bias, [None] * 4):
        _, lse, out32 = hip_simplicial_attention_forward(*ops, **kw, u=b[0], v_bias=b[1], w=b[2], gate=b[3],
                                                         precision="ieee_fp32")
        call = (go, *ops, out32, lse, *masks, *b, *[None] * 6, flags)
        results = []
        for fill in (0.0, float("nan")):
            real = torch.empty
            with pytest.MonkeyPatch.context() as mp:
                mp.setattr(hsa.torch, "empty", lambda *a, **k: real(*a, **k).fill_(fill)
                           if k.get("dtype") == torch.float32 else real(*a, **k))
                results.append(hsa._kernel_backward(*call))
        for want, got in zip(*results):
            assert (got is None) == (want is None)
            if got is not None:
                assert torch.equal(got, want)
        qp, kp = ~masks[0][:, None, :].expand(B, H, N), ~masks[1][:, None, :].expand(B, H, N)
        for g, pad in zip(results[1][:5], (qp, kp, kp, kp, kp)):
            assert not g[pad].any()


def test_writes_all_follows_the_route():
    """Only calls of the small fp32 kernel report that they write every element."""
    from matterformer_amd import _native

    lib = _native.lib()
    names = ("q", "k1", "v1", "k2", "v2", "grad_out", "out", "lse", "query_valid", "pair_key_valid", "dq", "dk1",
             "dv1", "dk2", "dv2")
    base = dict.fromkeys(names, 4096) | dict(batch=2, heads=2, tokens=32, head_dim=32, dtype=_native.MF_DTYPE_F32,
                                             grad_dtype=_native.MF_DTYPE_F32, grads_dtype=_native.MF_DTYPE_F32)
    for change, want in ((dict(), 1), (dict(tokens=33), 0), (dict(head_dim=36), 0), (dict(head_dim=30), 0),
                         (dict(dtype=_native.MF_DTYPE_BF16), 0), (dict(grad_dtype=_native.MF_DTYPE_BF16), 0),
                         (dict(dq=4100), 0), (dict(dk1=4100, dv1=4100), 1), (dict(angle_left=4096), 0),
                         (dict(message_left=4096), 0), (dict(dv2=None), 0)):
        assert lib.mf_simplicial_bwd_writes_all(_native.MfSimplicialBwdArgs(**(base | change))) == want, change
