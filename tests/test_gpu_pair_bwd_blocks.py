"""The pair-formulation backward at the edges of its blocks: 16-row tiles, 24 / 16 j per unit, 64 / 48 query and
key rows per block, and molecules whose units sum over several block triples, without a bias and with bf16 and fp32
bias terms.

Bars, normwise per gradient against float64 autograd on the same rounded inputs.  bf16 gradients: the rounding of
the result (2^-9 at most, 1.7e-3 over random mantissas) with the fp16 rounding of W, dS and P (2^-11 each, random
signs under sums) below it: 4e-3.  fp32 bias gradients: they sum fp32 dS, whose error is that of S (W rounded to
fp16: 2^-11 of |S| < 4, so P is off by 2e-3 of itself at most, 6e-4 over random roundings): 2e-3.
"""

import pytest
import torch

from matterformer_amd.workloads import random_simplicial
from test_gpu_simplicial_bwd import GRAD_NAMES, fp64_grads, hip_grads, logit_std, rel_err

pytestmark = pytest.mark.gpu

COUNTS = ([1, 2, 15], [16, 17, 24], [25, 47, 48], [49, 63, 64], [65, 80, 81], [97, 33], [146])


@pytest.mark.parametrize("bias_dtype", [None, torch.bfloat16, torch.float32], ids=["none", "bf16", "fp32"])
@pytest.mark.parametrize("counts", COUNTS, ids=lambda c: "n" + "-".join(map(str, c)))
def test_block_edges(cuda, counts, bias_dtype):
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
