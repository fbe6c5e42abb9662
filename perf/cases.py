"""The work that is timed and compared when this framework's kernels change.

Every case goes through entry points that a program calls: the projected 2-simplicial attention (forward, and
forward with backward), the attention layer, the geometry bias of a batch, radius attention in periodic cells,
kNN lists, and the whole trunk.  ``listed`` holds sizes from the framework's own configurations and its module
grid; ``draw`` gives sizes from the ranges around them.  Inputs are drawn on the GPU from the seed; ``exact``
restates each case in plain torch in 64 bits.

Masks are prefixes (a molecule's atoms first, padding after), as a padded batch of molecules has them.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from matterformer_amd.geometry import NonPeriodicGeometryAdapter
from matterformer_amd.geometry_bias import SimplicialGeometryBias
from matterformer_amd.geometry_ops import knn_graph, radius_attention, radius_mask
from matterformer_amd.hip_simplicial_attention import (
    hip_simplicial_attention_backward,
    hip_simplicial_attention_forward,
)
from matterformer_amd.simplicial_attention import TwoSimplicialAttention
from matterformer_amd.simplicial_types import SimplicialAttentionMask, SimplicialFactorizedBias
from matterformer_amd.trunk import AlternatingTrunk, TokenPacking

DEVICE = "cuda"
DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}
CORE = ("q", "k1", "v1", "k2", "v2")
BIAS = ("u", "v", "w", "gate")


# -- the cases ---------------------------------------------------------------------------------------------------
def _attention(name, *, train, dtype, molecules, batch, heads, head_dim, tokens, bias):
    return dict(name=name, kind="attention", train=train, dtype=dtype, molecules=molecules, batch=batch, heads=heads,
                head_dim=head_dim, tokens=tokens, bias=bias)


def listed():
    return [
        # one attention layer in the sampling of four molecules: the smallest call, where latency counts
        dict(name="layer_small", kind="layer", molecules="geom", batch=4, heads=8, head_dim=64, tokens=64,
             bias="float32"),
        # QM9 molecules in fp32, scored and trained
        _attention("qm9_fp32", train=False, dtype="float32", molecules="qm9", batch=128, heads=8, head_dim=32,
                   tokens=29, bias="none"),
        _attention("qm9_fp32_train", train=True, dtype="float32", molecules="qm9", batch=128, heads=8, head_dim=32,
                   tokens=29, bias="none"),
        # GEOM-Drugs molecules in bf16: a batch with the geometry bias (fp32, as the bias module returns it, and
        # the geometry pair mask), and a large batch without
        _attention("geom_bias", train=False, dtype="bfloat16", molecules="geom", batch=64, heads=8, head_dim=64,
                   tokens=181, bias="float32"),
        _attention("geom_large", train=False, dtype="bfloat16", molecules="geom", batch=512, heads=8, head_dim=64,
                   tokens=181, bias="none"),
        # the same molecules trained, without and with the geometry bias
        _attention("geom_train", train=True, dtype="bfloat16", molecules="geom", batch=64, heads=8, head_dim=64,
                   tokens=181, bias="none"),
        _attention("geom_bias_train", train=True, dtype="bfloat16", molecules="geom", batch=64, heads=8, head_dim=64,
                   tokens=181, bias="float32"),
        # the widest row of the module grid: every token valid, a bf16 bias that takes gradients
        _attention("dense_bias_train", train=True, dtype="bfloat16", molecules="dense", batch=4, heads=12,
                   head_dim=64, tokens=192, bias="bfloat16"),
        # the geometry bias of a training batch: pair features, the three pair MLPs, the gradients of their weights
        dict(name="geometry_bias_train", kind="geometry", train=True, molecules="geom", batch=64, tokens=181, heads=8,
             hidden=128, rbf=16),
        # radius attention in periodic MOF cells: the minimum-image cutoff mask and one attention over it
        dict(name="cells_radius", kind="cells", batch=32, atoms=512, heads=8, head_dim=64, cutoff=6.0),
        # the neighbour lists of a data set's molecules, in one call
        dict(name="knn_lists", kind="knn", batch=4096, atoms=181, k=16),
        # the 12-layer trunk with the geometry bias on a generation batch: one denoising step
        dict(name="trunk_step", kind="trunk", molecules="geom", batch=256, tokens=181, d_model=512, heads=8,
             layers=12, knn_k=32),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _mean_cube(molecules, tokens):
    if molecules == "dense":
        return tokens ** 3
    if molecules == "qm9":
        return sum(n ** 3 for n in range(9, 30)) / 21
    return 1.2 * 44 ** 3


def draw(rng):
    kind = rng.choice(("layer", "attention", "attention", "attention", "attention", "geometry", "cells", "knn", "trunk"))
    if kind == "layer":
        return dict(kind="layer", molecules="geom", batch=_log_int(rng, 1, 32), heads=rng.choice((4, 8, 12)),
                    head_dim=64, tokens=rng.randint(40, 120), bias=rng.choice(("none", "float32")))
    if kind == "attention":
        molecules = rng.choice(("qm9", "geom", "geom", "dense"))
        train = rng.random() < 0.5
        heads = rng.choice((4, 8, 8, 12))
        dtype = "float32" if molecules == "qm9" and rng.random() < 0.7 else "bfloat16"
        head_dim = rng.choice((32, 64)) if molecules == "qm9" else 64
        tokens = {"qm9": 29, "geom": rng.randint(90, 181), "dense": rng.randint(24, 192)}[molecules]
        bias = rng.choice(("none", "float32", "bfloat16"))
        if dtype == "float32" and bias != "none":
            bias = "float32"
        # at most the work of the largest listed case of the same direction
        cube = heads * head_dim * _mean_cube(molecules, tokens)
        most = (4 if train else 2) * 12 * 64 * 192 ** 3 / cube
        batch = _log_int(rng, 1, max(1, min(512, int(most) if molecules == "dense" else int(most / 2))))
        return dict(kind="attention", train=train, dtype=dtype, molecules=molecules, batch=batch, heads=heads,
                    head_dim=head_dim, tokens=tokens, bias=bias)
    if kind == "geometry":
        return dict(kind="geometry", train=rng.random() < 0.5, molecules=rng.choice(("qm9", "geom")),
                    batch=_log_int(rng, 2, 64), tokens=rng.randint(90, 181), heads=rng.choice((4, 8, 12)), hidden=128,
                    rbf=rng.choice((12, 16, 20)))
    if kind == "cells":
        return dict(kind="cells", batch=_log_int(rng, 1, 32), atoms=rng.randint(100, 512), heads=rng.choice((4, 8)),
                    head_dim=rng.choice((32, 64)), cutoff=round(rng.uniform(4.0, 7.0), 2))
    if kind == "knn":
        return dict(kind="knn", batch=_log_int(rng, 16, 4096), atoms=rng.randint(20, 181), k=rng.choice((8, 12, 16)))
    return dict(kind="trunk", molecules="geom", batch=_log_int(rng, 4, 192), tokens=rng.randint(100, 181),
                d_model=512, heads=8, layers=rng.choice((4, 8, 12)), knn_k=rng.choice((16, 32)))


# -- inputs ------------------------------------------------------------------------------------------------------
def _counts(case, seed):
    """Valid atoms of each molecule: QM9 uniform in 9..29, GEOM-Drugs round(44 + 12 z) in 10..tokens, dense all."""
    gen = torch.Generator().manual_seed(seed * 1009 + 7)
    B, N = case["batch"], case["tokens"]
    if case["molecules"] == "qm9":
        return torch.randint(9, min(N, 29) + 1, (B,), generator=gen)
    if case["molecules"] == "geom":
        z = torch.randn(B, generator=gen)
        return torch.clamp(torch.round(44.0 + 12.0 * z), 10, N).to(torch.int64)
    return torch.full((B,), N, dtype=torch.int64)


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed * 7919 + 13)


def _randn(gen, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=gen, device=DEVICE) * std).to(dtype)


def _valid(case, seed):
    counts = _counts(case, seed)
    valid = (torch.arange(case["tokens"])[None, :] < counts[:, None]).to(DEVICE)
    return counts.tolist(), valid


def _bias_terms(gen, case, valid):
    """u, v, w over the valid pairs (zero elsewhere, as the bias module masks them) and a gate per query in (0, 1)."""
    if case["bias"] == "none":
        return {}
    dt = DTYPES[case["bias"]]
    B, H, N = case["batch"], case["heads"], case["tokens"]
    pairs = (valid[:, :, None] & valid[:, None, :])[:, None].to(torch.float32)
    terms = {n: (_randn(gen, B, H, N, N, std=0.5) * pairs).to(dt) for n in ("u", "v", "w")}
    terms["gate"] = torch.sigmoid(_randn(gen, B, H, 1)).expand(B, H, N).contiguous().to(dt)
    return terms


def _prepare_attention(case, seed):
    gen = _generator(seed)
    B, H, N, D = case["batch"], case["heads"], case["tokens"], case["head_dim"]
    dt = DTYPES[case["dtype"]]
    counts, valid = _valid(case, seed)
    state = dict(case=case, counts=counts, valid=valid, pair_valid=None,
                 core=[_randn(gen, B, H, N, D, std=D ** -0.5, dtype=dt) for _ in CORE],
                 precision="ieee_fp32" if case["dtype"] == "float32" else "bf16_tc")
    state["bias"] = _bias_terms(gen, case, valid)
    if case["bias"] == "float32":  # the geometry pair mask comes with the bias module's terms
        state["pair_valid"] = valid[:, :, None] & valid[:, None, :]
    if case["train"]:
        state["grad_out"] = _randn(gen, B, H, N, D, dtype=dt)
    return state


def _run_attention(s):
    b = s["bias"]
    kwargs = dict(query_valid=s["valid"], pair_key_valid=s["valid"], pair_valid=s["pair_valid"],
                  precision=s["precision"])
    if b:
        kwargs.update(u=b["u"], v_bias=b["v"], w=b["w"], gate=b["gate"])
    if not s["case"]["train"]:
        return {"out": hip_simplicial_attention_forward(*s["core"], need_backward_state=False, **kwargs)[0]}
    out, lse, out_f32 = hip_simplicial_attention_forward(*s["core"], **kwargs)
    grads = hip_simplicial_attention_backward(s["grad_out"], *s["core"], out_f32, lse, **kwargs)
    result = {"out": out, "lse": lse}
    result.update(("d" + n, g) for n, g in zip(CORE, grads[:5]))
    if b:
        result.update(("d" + n, g) for n, g in zip(BIAS, grads[5:9]))
    return result


def _prepare_layer(case, seed):
    gen = _generator(seed)
    B, H, N, D = case["batch"], case["heads"], case["tokens"], case["head_dim"]
    counts, valid = _valid(case, seed)
    with torch.device(DEVICE):
        layer = TwoSimplicialAttention(H * D, H).to(torch.bfloat16).eval()
    for p in layer.parameters():
        p.data.copy_(_randn(gen, *p.shape, std=(H * D) ** -0.5))
    terms = _bias_terms(gen, case, valid)
    pair_valid = valid[:, :, None] & valid[:, None, :] if terms else None
    return dict(case=case, counts=counts, layer=layer, x=_randn(gen, B, N, H * D, dtype=torch.bfloat16),
                mask=SimplicialAttentionMask(query_valid=valid, pair_key_valid=valid, pair_valid=pair_valid),
                bias=SimplicialFactorizedBias(**terms) if terms else None)


def _run_layer(s):
    with torch.no_grad():
        return s["layer"](s["x"], attention_mask=s["mask"], factorized_bias=s["bias"])


def _bias_module(gen, heads, hidden, rbf):
    """A SimplicialGeometryBias on the GPU whose output layers are not zero (trained weights are not)."""
    module = SimplicialGeometryBias(heads, mode="factorized", edge_bias_hidden_dim=hidden, edge_bias_n_rbf=rbf)
    with torch.no_grad():  # the lazy layers take their sizes from a first call
        tiny = NonPeriodicGeometryAdapter()(torch.zeros(1, 2, 3))
        module.build_structured_bias_inputs(tiny, 2, sigma=torch.ones(1))
    module.to(DEVICE)
    for name, p in module.named_parameters():
        if "_mlp." in name:
            std = 0.3 if ".2." in name else p.shape[-1] ** -0.5 if p.ndim == 2 else 0.1
            p.data.copy_(_randn(gen, *p.shape, std=std))
    return module


def _prepare_geometry(case, seed):
    gen = _generator(seed)
    B, H, N = case["batch"], case["heads"], case["tokens"]
    counts, valid = _valid(case, seed)
    state = dict(case=case, counts=counts, adapter=NonPeriodicGeometryAdapter(),
                 module=_bias_module(gen, H, case["hidden"], case["rbf"]),
                 coords=_randn(gen, B, N, 3, std=math.sqrt(2.0)), pad=~valid,
                 sigma=torch.rand(B, generator=gen, device=DEVICE) * 2.0 + 0.05)
    if case["train"]:  # what the attention's backward hands back: gradients at the valid pairs
        pairs = (valid[:, :, None] & valid[:, None, :])[:, None]
        state["grads"] = [_randn(gen, B, H, N, N) * pairs for _ in range(3)]
    return state


def _run_geometry(s):
    with torch.set_grad_enabled(s["case"]["train"]):
        geom = s["adapter"](s["coords"], s["pad"])
        bias = s["module"].build_structured_bias_inputs(geom, s["case"]["tokens"], pad_mask=s["pad"],
                                                        sigma=s["sigma"])[0]
    result = {"u": bias.u, "v": bias.v, "w": bias.w, "gate": bias.gate}
    if s["case"]["train"]:
        params = [(n, p) for n, p in s["module"].named_parameters() if "_mlp." in n]
        grads = torch.autograd.grad([bias.u, bias.v, bias.w], [p for _, p in params], s["grads"])
        result.update((n.replace(".", "_"), g) for (n, _), g in zip(params, grads))
    return result


def _prepare_cells(case, seed):
    gen = _generator(seed)
    B, N, H, D = case["batch"], case["atoms"], case["heads"], case["head_dim"]
    rand = lambda *shape: torch.rand(*shape, generator=gen, device=DEVICE)  # noqa: E731
    lengths = 15.0 + 15.0 * rand(B, 3)
    angles = (80.0 + 20.0 * rand(B, 3)) * math.pi / 180.0
    return dict(case=case, frac=rand(B, N, 3), lattice=torch.cat([lengths.log(), angles.cos()], dim=-1),
                qkv=[_randn(gen, B, H, N, D, std=0.125, dtype=torch.bfloat16) for _ in range(3)])


def _run_cells(s):
    bits, blocks = radius_mask(s["frac"], s["case"]["cutoff"], lattice=s["lattice"])
    return {"bits": bits, "blocks": blocks, "out": radius_attention(*s["qkv"], bits, blocks)}


def _prepare_knn(case, seed):
    gen = _generator(seed)
    return dict(case=case, coords=_randn(gen, case["batch"], case["atoms"], 3, std=math.sqrt(2.0)))


def _run_knn(s):
    idx, dist = knn_graph(s["coords"], s["case"]["k"])
    return {"idx": idx, "dist": dist}


def _prepare_trunk(case, seed):
    gen = _generator(seed)
    B, N, C = case["batch"], case["tokens"], case["d_model"]
    counts, valid = _valid(case, seed)
    with torch.device(DEVICE):
        trunk = AlternatingTrunk(C, case["heads"], case["layers"], knn_k=case["knn_k"])
    trunk.blocks.to(torch.bfloat16)
    for name, p in trunk.named_parameters():
        std = 0.05 if "ada_ln" in name else p.shape[-1] ** -0.5 if p.ndim == 2 else 0.02
        p.data.copy_(_randn(gen, *p.shape, std=std))
    trunk.geometry_adapter = NonPeriodicGeometryAdapter()
    trunk.simplicial_geometry_bias = _bias_module(gen, case["heads"], 128, 16)
    trunk.eval()
    # a sampler keeps the packing of its batch over the denoising steps
    return dict(case=case, counts=counts, trunk=trunk, pad=~valid, packing=TokenPacking(~valid),
                x=_randn(gen, B, N, C, dtype=torch.bfloat16), cond=_randn(gen, B, C, dtype=torch.bfloat16),
                coords=_randn(gen, B, N, 3, std=math.sqrt(2.0)),
                sigma=torch.rand(B, generator=gen, device=DEVICE) * 2.0 + 0.05)


def _run_trunk(s):
    with torch.no_grad():
        return s["trunk"](s["x"], s["cond"], s["coords"], s["pad"], sigma=s["sigma"], packing=s["packing"])


PREPARE = dict(attention=_prepare_attention, layer=_prepare_layer, geometry=_prepare_geometry, cells=_prepare_cells,
               knn=_prepare_knn, trunk=_prepare_trunk)
RUN = dict(attention=_run_attention, layer=_run_layer, geometry=_run_geometry, cells=_run_cells, knn=_run_knn,
           trunk=_run_trunk)


def prepare(case, seed):
    return PREPARE[case["kind"]](case, seed)


def run(state):
    return RUN[state["case"]["kind"]](state)


# -- what a pass cannot do without -------------------------------------------------------------------------------
def _attention_work(case, rows, squares, cubes):
    """rows, squares, cubes: sums of n, n^2, n^3 over the molecules."""
    B, H, N, D = case["batch"], case["heads"], case["tokens"], case["head_dim"]
    item = 2 if case.get("dtype", "bfloat16") == "bfloat16" else 4
    train = case.get("train", False)
    flops = 4 * H * D * cubes
    moved = 5 * rows * H * D * item + B * H * N * D * item
    bias = {"none": 0, "float32": 4, "bfloat16": 2}[case["bias"]]
    moved += 3 * H * squares * bias
    if train:  # five products of n^3 D beside the forward's two; gradients of every operand, written whole
        flops += 10 * H * D * cubes
        moved += rows * H * D * item + 5 * B * H * N * D * item + 4 * B * H * N
        moved += 3 * B * H * N * N * bias
    return flops, moved


def work(case):
    kind = case["kind"]
    if kind == "knn":
        B, N, k = case["batch"], case["atoms"], case["k"]
        return {"bytes": B * N * (12 + 8 * k), "flops": 8 * B * N * N}
    if kind == "cells":
        B, N, H, D = case["batch"], case["atoms"], case["heads"], case["head_dim"]
        near = min(1.0, 4.19 * case["cutoff"] ** 3 / 22.5 ** 3)  # the share of a cell within the cutoff
        return {"bytes": B * N * (12 + 4 * H * D * 2 + N / 8), "flops": 4 * B * H * D * N * N * near + 16 * B * N * N}
    counts = _counts(case, 0).double()
    rows, squares, cubes = (float((counts ** p).sum()) for p in (1, 2, 3))
    if kind == "attention":
        flops, moved = _attention_work(case, rows, squares, cubes)
        return {"bytes": moved, "flops": flops}
    if kind == "layer":
        C = case["heads"] * case["head_dim"]
        flops, _ = _attention_work(case, rows, squares, cubes)
        bias = 12 * case["heads"] * squares if case["bias"] != "none" else 0
        return {"bytes": 12 * C * C + 4 * case["batch"] * case["tokens"] * C + bias, "flops": flops + 12 * C * C * rows}
    if kind == "geometry":
        H, hidden, N, B = case["heads"], case["hidden"], case["tokens"], case["batch"]
        per_pair = 2 * hidden * (2 * (3 + case["rbf"]) + case["rbf"] + 3 * H)
        moved = 12 * rows + 12 * B * H * N * N  # coordinates; u, v, w written whole
        flops = per_pair * squares
        if case["train"]:  # the upstream gradients at the valid pairs; both layers' weight gradients, dh, layer 1 again
            moved += 12 * H * squares
            flops *= 3
        return {"bytes": moved, "flops": flops}
    C, H, L, k = case["d_model"], case["heads"], case["layers"], case["knn_k"]
    simp, local = (L + 1) // 2, L // 2
    flops = (28 * simp + 24 * local) * C * C * rows + 12 * L * C * C * case["batch"]
    flops += simp * 4 * C * cubes + local * 4 * C * (k + 1) * rows
    moved = 4 * case["batch"] * case["tokens"] * C + 2 * C * C * (20 * simp + 18 * local)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """About four times the error against ``exact`` that the kernels show: 32-bit sums 1e-6, bf16 results 2.4e-3,
    the layer (bf16 projections around the attention) 4.7e-3, the whole trunk 1.2e-2."""
    kind = case["kind"]
    if kind == "knn":
        return "exact"
    if kind == "geometry" or case.get("dtype") == "float32":
        return {"rel": 5e-6, "max": 5e-4}
    if kind == "layer":
        return {"rel": 2e-2, "max": 0.3}
    if kind == "trunk":
        return {"rel": 3e-2, "max": 0.5}
    return {"rel": 1e-2, "max": 0.2}


# -- the same results in 64 bits, in plain torch -----------------------------------------------------------------
def _core64(q, k1, v1, k2, v2, bias=None):
    """One molecule's attention (H, n, D) and its logsumexp (H, n); bias: u, v, w (H, n, n) and gate (H, n)."""
    H, n, D = q.shape
    a = (q[:, :, None, :] * k1[:, None, :, :]).reshape(H, n * n, D)
    s = torch.matmul(a, k2.transpose(1, 2).contiguous()).view(H, n, n, n)
    if bias is not None:
        u, v, w, gate = bias
        s = s + gate[:, :, None, None] * (u[:, :, :, None] + v[:, :, None, :] + w[:, None, :, :])
    lse = torch.logsumexp(s.view(H, n, n * n), dim=-1)
    p = torch.exp(s - lse[:, :, None, None])
    t = torch.matmul(p.view(H, n * n, n), v2).view(H, n, n, D)
    return (t * v1[:, None]).sum(dim=2), lse


def _exact_attention(case, s):
    out, lse = torch.zeros_like(s["core"][0], dtype=torch.float64), None
    result = {"out": out}
    names = CORE + (BIAS if s["bias"] else ())
    whole = dict(zip(CORE, s["core"]), **s["bias"])
    if case["train"]:
        lse = result["lse"] = torch.zeros(out.shape[:3], dtype=torch.float64, device=DEVICE)
        for n in names:
            result["d" + n] = torch.zeros_like(whole[n], dtype=torch.float64)
    for b, n in enumerate(s["counts"]):
        cut = {name: (t[b, :, :n, :n] if name in ("u", "v", "w") else t[b, :, :n]).double() for name, t in whole.items()}
        leaves = [cut[name].requires_grad_(case["train"]) for name in names]
        o, l = _core64(*leaves[:5], bias=leaves[5:] or None)
        out[b, :, :n] = o.detach()
        if case["train"]:
            lse[b, :, :n] = l.detach()
            for name, g in zip(names, torch.autograd.grad(o, leaves, s["grad_out"][b, :, :n].double())):
                at = result["d" + name][b]
                (at[:, :n, :n] if name in ("u", "v", "w") else at[:, :n]).copy_(g)
    return result


def _linear64(x, weight, bias):
    return torch.matmul(x, weight.double().t()) + bias.double()


def _heads64(x, H):
    return x.view(x.shape[0], H, -1).transpose(0, 1)


def _layer64(attn, x, H, bias):
    """TwoSimplicialAttention on one molecule's rows (n, C)."""
    q, k1, v1, k2, v2 = (_heads64(t, H) for t in _linear64(x, attn.in_proj.weight, attn.in_proj.bias).chunk(5, dim=-1))
    out, _ = _core64(q * q.shape[-1] ** -0.5, k1, v1, k2, v2, bias)
    return _linear64(out.transpose(0, 1).reshape(x.shape[0], -1), attn.out_proj.weight, attn.out_proj.bias)


def _exact_layer(case, s):
    result = torch.zeros_like(s["x"], dtype=torch.float64)
    # rows past a molecule's end: attention gives 0 there, out_proj its bias
    result += s["layer"].out_proj.bias.double()
    fb = s["bias"]
    for b, n in enumerate(s["counts"]):
        bias = None
        if fb is not None:
            bias = [t[b, :, :n, :n].double() for t in (fb.u, fb.v, fb.w)] + [fb.gate[b, :, :n].double()]
        result[b, :n] = _layer64(s["layer"], s["x"][b, :n].double(), case["heads"], bias)
    return result


def _geometry64(module, params, coords, sigma):
    """u, v, w (H, n, n) and the gate (H,) of one molecule's coordinates (n, 3)."""
    n = coords.shape[0]
    rms = torch.sqrt(coords.square().sum(-1).mean().clamp_min(1e-8))
    delta = coords[:, None, :] - coords[None, :, :]
    dist = torch.sqrt(delta.square().sum(-1))
    centers = module._edge_rbf_centers.double()
    rbf = torch.exp(-module._edge_rbf_gamma.double() * (dist[..., None] / rms - centers).square())
    spoke = torch.cat([delta, rbf], dim=-1)
    off = 1.0 - torch.eye(n, dtype=torch.float64, device=coords.device)
    terms = []
    for name, feats in (("spoke_bias_u_mlp", spoke), ("spoke_bias_v_mlp", spoke), ("pair_bias_w_mlp", rbf)):
        h = F.silu(torch.matmul(feats.reshape(n * n, -1), params[name + ".0.weight"].t()) + params[name + ".0.bias"])
        y = torch.matmul(h, params[name + ".2.weight"].t()) + params[name + ".2.bias"]
        terms.append(y.t().reshape(-1, n, n) * off)
    alpha = F.softplus(module.noise_gate_alpha_raw.detach().double()).view(-1)
    gate = torch.sigmoid(-alpha * torch.log(sigma) + module.noise_gate_beta.detach().double().view(-1))
    return terms, gate


def _exact_geometry(case, s):
    B, H, N = case["batch"], case["heads"], case["tokens"]
    module = s["module"]
    params = {n: p.detach().double().requires_grad_(case["train"]) for n, p in module.named_parameters() if "_mlp." in n}
    result = {n: torch.zeros(B, H, N, N, dtype=torch.float64, device=DEVICE) for n in ("u", "v", "w")}
    result["gate"] = torch.zeros(B, H, N, dtype=torch.float64, device=DEVICE)
    grads = {n: torch.zeros_like(p) for n, p in params.items()}
    for b, n in enumerate(s["counts"]):
        terms, gate = _geometry64(module, params, s["coords"][b, :n].double(), s["sigma"][b].double())
        for name, t in zip(("u", "v", "w"), terms):
            result[name][b, :, :n, :n] = t.detach()
        result["gate"][b] = gate[:, None]
        if case["train"]:
            ups = [g[b, :, :n, :n].double() for g in s["grads"]]
            for name, g in zip(params, torch.autograd.grad(terms, list(params.values()), ups)):
                grads[name] += g
    if case["train"]:
        result.update((n.replace(".", "_"), g) for n, g in grads.items())
    return result


def _cell64(lattice):
    """Rows of the cell matrices (B, 3, 3): a along x, b in the xy plane."""
    lengths = torch.exp(lattice[:, :3])
    ca, cb, cg = lattice[:, 3:].unbind(dim=-1)
    sg = torch.sqrt(1.0 - cg.square())
    cell = torch.zeros(lattice.shape[0], 3, 3, dtype=torch.float64, device=lattice.device)
    cell[:, 0, 0] = lengths[:, 0]
    cell[:, 1, 0], cell[:, 1, 1] = lengths[:, 1] * cg, lengths[:, 1] * sg
    cell[:, 2, 0], cell[:, 2, 1] = lengths[:, 2] * cb, lengths[:, 2] * (ca - cb * cg) / sg
    cell[:, 2, 2] = torch.sqrt(lengths[:, 2].square() - cell[:, 2, 0].square() - cell[:, 2, 1].square())
    return cell


def _exact_cells(case, s):
    cells = _cell64(s["lattice"].double())
    q, k, v = s["qkv"]
    out = torch.zeros_like(q, dtype=torch.float64)
    for b in range(case["batch"]):
        frac = s["frac"][b].double()
        delta = frac[:, None, :] - frac[None, :, :]
        d2 = torch.full(delta.shape[:2], math.inf, dtype=torch.float64, device=DEVICE)
        for image in range(27):
            shift = torch.tensor([image // 9 - 1, image // 3 % 3 - 1, image % 3 - 1], dtype=torch.float64, device=DEVICE)
            d2 = torch.minimum(d2, torch.matmul(delta + shift, cells[b]).square().sum(-1))
        logits = torch.matmul(q[b].double(), k[b].double().transpose(1, 2).contiguous()) * q.shape[-1] ** -0.5
        p = torch.softmax(logits.masked_fill(d2 > case["cutoff"] ** 2, -math.inf), dim=-1)
        out[b] = torch.matmul(p, v[b].double())
    return {"bits": None, "blocks": None, "out": out}


def _exact_knn(case, s):
    """The k smallest distances of every atom (the order of the lists is fixed in fp32: no 64-bit answer)."""
    parts = []
    for c in s["coords"].split(256):
        c = c.double()
        d2 = (c[:, :, None, :] - c[:, None, :, :]).square().sum(-1)
        d2.diagonal(dim1=1, dim2=2).fill_(math.inf)
        parts.append(torch.sqrt(torch.topk(d2, min(case["k"], c.shape[1]), dim=-1, largest=False).values))
    return {"idx": None, "dist": torch.cat(parts)}


def _nearest(coords, k):
    """(n, n) bool: j among the k nearest of i, or i itself."""
    n = coords.shape[0]
    d = coords[:, None, :] - coords[None, :, :]
    d2 = (d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2]
    d2.fill_diagonal_(-1.0)
    order = torch.sort(d2, dim=-1, stable=True).indices[:, :k + 1]
    return torch.zeros(n, n, dtype=torch.bool, device=coords.device).scatter_(1, order, True)


def _exact_trunk(case, s):
    H, C = case["heads"], case["d_model"]
    trunk, counts = s["trunk"], s["counts"]
    module = trunk.simplicial_geometry_bias
    params = {n: p.detach().double() for n, p in module.named_parameters() if "_mlp." in n}
    rows = torch.cat([s["x"][b, :n] for b, n in enumerate(counts)]).double()
    mol = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts)).to(DEVICE)
    cond = F.silu(s["cond"].double())
    bias, near = [], []
    for b, n in enumerate(counts):
        terms, gate = _geometry64(module, params, s["coords"][b, :n].double(), s["sigma"][b].double())
        bias.append(terms + [gate[:, None].expand(H, n)])
        near.append(_nearest(s["coords"][b, :n], case["knn_k"]))

    def normed(x, eps, shift, scale):
        return F.layer_norm(x, (C,), eps=eps) * (1.0 + scale[mol]) + shift[mol]

    for block in trunk.blocks:
        lin = block.ada_ln[-1]
        shift_a, scale_a, gate_a, shift_m, scale_m, gate_m = _linear64(cond, lin.weight, lin.bias).chunk(6, dim=-1)
        parts = normed(rows, block.norm1.eps, shift_a, scale_a).split(counts)
        if block.attn_type == "simplicial":
            attn = torch.cat([_layer64(block.attn, x, H, bias[b]) for b, x in enumerate(parts)])
        else:
            mha, done = block.attn.attn, []
            for b, x in enumerate(parts):
                q, k, v = (_heads64(t, H) for t in _linear64(x, mha.in_proj_weight, mha.in_proj_bias).chunk(3, dim=-1))
                logits = torch.matmul(q, k.transpose(1, 2).contiguous()) * q.shape[-1] ** -0.5
                p = torch.softmax(logits.masked_fill(~near[b], -math.inf), dim=-1)
                o = torch.matmul(p, v).transpose(0, 1).reshape(x.shape[0], C)
                done.append(_linear64(o, mha.out_proj.weight, mha.out_proj.bias))
            attn = torch.cat(done)
        rows = rows + gate_a[mol] * attn
        h = normed(rows, block.norm2.eps, shift_m, scale_m)
        h = F.gelu(_linear64(h, block.mlp.fc1.weight, block.mlp.fc1.bias), approximate="tanh")
        rows = rows + gate_m[mol] * _linear64(h, block.mlp.fc2.weight, block.mlp.fc2.bias)
    out = torch.zeros_like(s["x"], dtype=torch.float64)
    for b, x in enumerate(rows.split(counts)):
        out[b, :counts[b]] = x
    return out


EXACT = dict(attention=_exact_attention, layer=_exact_layer, geometry=_exact_geometry, cells=_exact_cells,
             knn=_exact_knn, trunk=_exact_trunk)


def exact(case, seed):
    if case["kind"] == "knn" and case["k"] >= case["atoms"]:
        return None
    state = prepare(case, seed)
    with torch.set_grad_enabled(bool(case.get("train"))):
        return EXACT[case["kind"]](case, state)
