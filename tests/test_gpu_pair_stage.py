"""The pair kernel's staging of bias terms and pair-valid bits at the edges of what it splits: 32, 64 and 80 keys (row
groups, the first 64 columns and those past them, one key block) with the bias, 64 and 128 without, odd counts (a
padding row in the last row pair), one and two query groups, masks that are no prefix, every bias dtype.

Bars as for the 16-bit forward elsewhere, against float64 on the same 16-bit inputs: normwise 2e-2 and every valid
query row within 3e-2 of its own norm (bf16 output rounding 2^-9 a component, fp16 products and probabilities
2^-11 a rounding; a wrong bias row or pair bit moves a row by its own size)."""

import pytest
import torch

from matterformer_amd.workloads import random_simplicial
from test_gpu_simplicial_bias import logit_std, make_terms, oracle, rel_err, row_errors, run

pytestmark = pytest.mark.gpu

CASES = [
    # counts, head_dim, bias dtype (None: no bias), pair_valid
    ([1, 2, 3], 64, torch.float32, True),
    ([15, 16, 17], 32, torch.bfloat16, True),
    ([31, 32, 33], 64, torch.float32, False),
    ([47, 49, 48], 40, torch.float16, True),
    ([63, 64, 65], 64, torch.float32, True),
    ([65, 66, 64], 64, torch.bfloat16, True),
    ([79, 80, 81], 64, torch.float32, True),
    ([80, 77], 32, torch.float16, False),
    ([97, 160, 161], 64, torch.float32, True),
    ([63, 64, 65], 64, None, True),
    ([127, 128, 129], 64, None, True),
]


@pytest.mark.parametrize("prefix", [True, False], ids=["prefix", "scattered"])
@pytest.mark.parametrize("counts,D,bias_dtype,pairs", CASES,
                         ids=lambda v: "-".join(map(str, v)) if isinstance(v, list) else str(v).replace("torch.", ""))
def test_staging_edges(cuda, counts, D, bias_dtype, pairs, prefix):
    B, H, N = len(counts), 2, max(counts)
    case = list(random_simplicial(B, H, N, D, seed=N + D + 3, counts=counts, pair_drop=0.2 if pairs else 0.0,
                                  std=logit_std(D)))
    if not prefix:  # the same numbers of valid tokens, the padding spread between them
        gen = torch.Generator().manual_seed(N)
        for b in range(B):
            perm = torch.randperm(N, generator=gen)
            case[5][b] = case[5][b][perm]
            case[6][b] = case[6][b][perm]
    if pairs:  # every key row keeps its own pair, so no query is without pairs
        case[7] = case[7] | torch.eye(N, dtype=torch.bool)
    terms = {} if bias_dtype is None else make_terms(B, H, N, D, seed=N * 7 + D)
    out, _, _ = run(case, terms, cuda, torch.bfloat16, "bf16_tc", bias_dtype=bias_dtype)
    ref, _ = oracle(case, terms, torch.bfloat16, bias_dtype=bias_dtype)
    got = out.float().cpu().numpy()
    assert rel_err(got, ref) <= 2e-2
    assert row_errors(got, ref, case[5]).max() <= 3e-2
