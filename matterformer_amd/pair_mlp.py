"""The factorized geometry-bias MLPs on the GPU: SimplicialGeometryBias._compute_factorized_terms
(src/matterformer/models/transformer.py:702-717) as one mf_pair_mlp_bias pass over the valid pairs, and, when
the MLP weights take gradients, its weight backward as one mf_pair_mlp_bias_bwd pass (an autograd Function).

Served: GPU features, fp32 weights and features, materialised LazyLinear layers (their first call runs the
torch formulation, which draws their weights in the reference's order), rbf <= 29, hidden a multiple of 16
<= 256, heads <= 16, and with use_periodic_features on periodic features (Fourier terms of the pair delta and
the cell's global features, transformer.py:641-652) at most 80 spoke inputs; under autograd also rbf <= 28,
hidden <= 128, non-periodic features and features that take no gradient.  Everything else takes the torch
formulation.
"""

from __future__ import annotations

import torch
from torch.nn.parameter import UninitializedParameter

from matterformer_amd import _native


def _mlps(module):
    return module.spoke_bias_u_mlp, module.spoke_bias_v_mlp, module.pair_bias_w_mlp


def _weights(module) -> list[torch.Tensor]:
    """W1, b1, W2, b2 of the u, v, w MLPs, in that order (12 tensors)."""
    out = []
    for mlp in _mlps(module):
        first, last = mlp[0], mlp[2]
        out += [first.weight, first.bias, last.weight, last.bias]
    return out


def _trains(module, geom_features) -> bool:
    g = geom_features
    return torch.is_grad_enabled() and (any(prm.requires_grad for m in _mlps(module) for prm in m.parameters())
                                        or g.pair_delta.requires_grad or g.pair_dist_norm.requires_grad)


def _periodic(module, geom_features) -> bool:
    return bool(module.use_periodic_features) and geom_features.kind == "periodic"


def serves(module, geom_features) -> bool:
    g = geom_features
    if g.pair_delta.device.type != "cuda":
        return False
    mlps = _mlps(module)
    params = [prm for m in mlps for prm in m.parameters()]
    if any(isinstance(prm, UninitializedParameter) for prm in params):
        return False
    if not isinstance(mlps[0][1], torch.nn.SiLU):
        return False
    R = module.edge_bias_n_rbf
    hidden = mlps[0][0].out_features
    if not (1 <= R <= 29 and hidden % 16 == 0 and 16 <= hidden <= 256 and 1 <= module.n_heads <= 16):
        return False
    if any(m[0].out_features != hidden or m[0].bias is None or m[2].bias is None for m in mlps):
        return False
    per = _periodic(module, g)
    nf = int(module._edge_freqs.numel()) if per else 0
    fs, fp = 3 + R + (6 * nf + 6 if per else 0), R + (6 if per else 0)
    if mlps[0][0].in_features != fs or mlps[1][0].in_features != fs or mlps[2][0].in_features != fp:
        return False
    if per and (fs > 80 or fp > 36 or g.global_geom.shape != (g.pair_delta.shape[0], 6)
                or g.global_geom.dtype != torch.float32):
        return False
    tensors = [g.pair_delta, g.pair_dist_norm] + params
    if not all(t.dtype == torch.float32 for t in tensors):
        return False
    if _trains(module, g):
        # the weight backward: non-periodic features without gradient, R <= 28, hidden <= 128
        if per or g.pair_delta.requires_grad or g.pair_dist_norm.requires_grad:
            return False
        return R <= 28 and hidden <= 128
    return True


def _forward_args(module, delta, dnorm, mask, centers, gamma, weights, outs, periodic=None):
    """periodic: None, or (freqs [nf], global_geom [B, 6]) fp32 contiguous."""
    B, N = delta.shape[:2]
    fields = {}
    if periodic is not None:
        fields.update(n_freqs=int(periodic[0].numel()), freqs=periodic[0].data_ptr(),
                      global_geom=periodic[1].data_ptr())
    for idx, name in enumerate("uvw"):
        for k, key in enumerate(("w1", "b1", "w2", "b2")):
            fields[f"{name}_{key}"] = weights[4 * idx + k].data_ptr()
    return _native.MfPairMlpArgs(
        pair_delta=delta.data_ptr(), pair_dist_norm=dnorm.data_ptr(), pair_mask=mask.data_ptr(),
        rbf_centers=centers.data_ptr(), rbf_gamma=gamma,
        u_out=_native.ptr(outs[0]), v_out=_native.ptr(outs[1]), w_out=_native.ptr(outs[2]),
        batch=B, atoms=N, rbf=int(centers.numel()), hidden=int(weights[0].shape[0]), heads=int(weights[2].shape[0]),
        **fields)


def _inputs(module, geom_features, atom_pad):
    g = geom_features
    dev = g.pair_delta.device
    delta = g.pair_delta.detach().contiguous()
    dnorm = g.pair_dist_norm.detach().contiguous()
    mask = g.pair_mask
    if mask.dtype != torch.bool:
        mask = mask.to(torch.uint8) != 0
    if atom_pad is not None:
        keep = ~atom_pad
        mask = mask & (keep[:, :, None] & keep[:, None, :])
    mask = mask.contiguous().view(torch.uint8)  # a bool's byte is 0 or 1
    centers = module._edge_rbf_centers.to(device=dev, dtype=torch.float32).contiguous()
    return delta, dnorm, mask, centers, float(module._edge_rbf_gamma_value)


def _run_forward(module, delta, dnorm, mask, centers, gamma, weights, periodic=None):
    B, N = delta.shape[:2]
    H = int(weights[2].shape[0])
    dev = delta.device
    outs = [torch.empty(B, H, N, N, device=dev, dtype=torch.float32) for _ in range(3)]
    args = _forward_args(module, delta, dnorm, mask, centers, gamma, weights, outs, periodic)
    with torch.cuda.device(dev):
        _native.check(_native.lib().mf_pair_mlp_bias(args, _native.current_stream(dev)), "mf_pair_mlp_bias")
    return outs


class _PairMlpFunction(torch.autograd.Function):
    """u, v, w from mf_pair_mlp_bias; the gradients of the 12 MLP weights from mf_pair_mlp_bias_bwd."""

    @staticmethod
    def forward(ctx, module, delta, dnorm, mask, centers, gamma, *weights):
        ws = [w.detach().contiguous() for w in weights]
        outs = _run_forward(module, delta, dnorm, mask, centers, gamma, ws)
        ctx.save_for_backward(delta, dnorm, mask, centers, *ws)
        ctx.gamma = gamma
        ctx.module = module
        return tuple(outs)

    @staticmethod
    def backward(ctx, gu, gv, gw):
        delta, dnorm, mask, centers, *ws = ctx.saved_tensors
        dev = delta.device
        B, N = delta.shape[:2]
        H = int(ws[2].shape[0])
        hidden = int(ws[0].shape[0])
        ups = []
        for gt in (gu, gv, gw):
            ups.append(torch.zeros(B, H, N, N, device=dev, dtype=torch.float32) if gt is None
                       else gt.float().contiguous())
        grads = [torch.empty_like(w) for w in ws]
        lib = _native.lib()
        nbytes = int(lib.mf_pair_mlp_bias_bwd_workspace_size(hidden))
        workspace = torch.empty(nbytes, device=dev, dtype=torch.uint8)
        fields = {}
        for idx, name in enumerate("uvw"):
            for k, key in enumerate(("dw1", "db1", "dw2", "db2")):
                fields[f"{name}_{key}"] = grads[4 * idx + k].data_ptr()
        args = _native.MfPairMlpBwdArgs(
            fwd=_forward_args(ctx.module, delta, dnorm, mask, centers, ctx.gamma, ws, (None, None, None)),
            u_grad=ups[0].data_ptr(), v_grad=ups[1].data_ptr(), w_grad=ups[2].data_ptr(),
            workspace=workspace.data_ptr(), workspace_bytes=nbytes, **fields)
        with torch.cuda.device(dev):
            _native.check(lib.mf_pair_mlp_bias_bwd(args, _native.current_stream(dev)), "mf_pair_mlp_bias_bwd")
        return (None, None, None, None, None, None, *grads)


def factorized_terms(module, geom_features, atom_pad=None):
    """(u, v, w) [B, H, N, N] fp32, diagonal and invalid pairs zero (the rows and columns of the atoms that
    atom_pad [B, N] bool marks too); differentiable in the MLP weights when they take gradients."""
    delta, dnorm, mask, centers, gamma = _inputs(module, geom_features, atom_pad)
    weights = _weights(module)
    if _trains(module, geom_features):
        return _PairMlpFunction.apply(module, delta, dnorm, mask, centers, gamma, *weights)
    periodic = None
    if _periodic(module, geom_features):
        dev = delta.device
        periodic = (module._edge_freqs.to(device=dev, dtype=torch.float32).contiguous(),
                    geom_features.global_geom.detach().to(device=dev, dtype=torch.float32).contiguous())
    with torch.no_grad():
        return tuple(_run_forward(module, delta, dnorm, mask, centers, gamma,
                                  [w.contiguous() for w in weights], periodic))
