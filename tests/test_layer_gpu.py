"""GPU parity of the GatedDeltaLayer kernels (producer, gated RMSNorm) and of
the whole layer, through the C ABI, against the CPU restatement in
oracle/layer_reference.py evaluated in fp64 on the same (dtype-rounded) inputs.

Bars: rel-L2 <= 1e-4 with fp32 activations, <= 1e-2 with bf16 activations,
for every output and every gradient (inputs and parameters)."""
import pytest
import torch

from oracle import kda_reference as R
from oracle import layer_reference as LR

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = {torch.float32: 1e-4, torch.bfloat16: 1e-2}


def _rel(a, b):
    return R.rel_l2(a.detach().cpu().double(), b.detach().cpu().double())


def _check(errs, tol, case):
    print(case, {k: f"{v:.2e}" for k, v in errs.items()}, flush=True)
    bad = {k: v for k, v in errs.items() if not (v <= tol)}
    assert not bad, f"{case}: {bad} above {tol}"


def _prod_inputs(B, T, H, D, dtype, seed, bias=True):
    g = torch.Generator().manual_seed(seed)
    HD = H * D
    r = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    acts = dict(qkv=r(B, T, 3 * HD), xf=r(B, T, HD), xb=r(B, T, H))
    acts = {n: t.to(dtype) for n, t in acts.items()}
    params = dict(conv_w=torch.rand(3, HD, 4, generator=g) - 0.5,
                  conv_b=0.1 * r(3, HD) if bias else None, dt_bias=0.1 * r(HD),
                  A_log=torch.log(1 + 15 * torch.rand(H, generator=g)))
    cots = dict(dq=r(B, T, H, D).to(dtype), dk=r(B, T, H, D).to(dtype), dv=r(B, T, H, D).to(dtype),
                dg=r(B, T, H, D), dbeta=r(B, T, H).to(dtype))
    return acts, params, cots


def _prod_reference(acts, params, cots, H, D, mult):
    HD = H * D
    leaves = {n: t.double().requires_grad_() for n, t in acts.items()}
    leaves.update({n: t.double().requires_grad_() for n, t in params.items() if t is not None})
    xq, xk, xv = leaves["qkv"].split(HD, -1)
    outs = LR.producer_from_projections(xq, xk, xv, leaves["xf"], leaves["xb"], leaves["conv_w"],
                                        leaves.get("conv_b"), leaves["dt_bias"], leaves["A_log"], H, D, mult)
    loss = sum((o * cots[n].double()).sum() for o, n in zip(outs, ("dq", "dk", "dv", "dg", "dbeta")))
    loss.backward()
    return outs, {n: t.grad for n, t in leaves.items()}


PRODUCER_CASES = [
    # B, T, H, D, dtype, bias, beta_mult
    (2, 37, 3, 64, torch.float32, True, 1.0),      # H*D = 192: one wave, a quarter of its lanes idle
    (1, 100, 12, 64, torch.float32, True, 1.0),    # H*D = 768: three waves per row
    (2, 5, 2, 32, torch.float32, True, 1.0),       # T shorter than a strip
    (1, 1, 6, 64, torch.float32, True, 1.0),       # T = 1
    (1, 70, 16, 128, torch.float32, True, 1.0),    # H*D = 2048: eight waves
    (3, 33, 4, 32, torch.float32, False, 2.0),     # no conv bias, allow_neg_eigval
    (2, 77, 12, 64, torch.bfloat16, True, 1.0),
    (1, 40, 6, 64, torch.bfloat16, False, 2.0),
    # enough row segments (>= 16) that the parameter-gradient column sums run
    # as two passes over row slices
    (2, 300, 4, 64, torch.float32, True, 1.0),
    (4, 260, 3, 64, torch.bfloat16, True, 1.0),
    (2, 37, 8, 96, torch.float32, True, 1.0),      # the SSv2 layer's 8 heads x 96
    # short sequences, several in one workgroup of the backward: 3 of 10 tokens
    # with two over, 2 of 16, up to 32 of one; 17 tokens are a segment of their own
    (386, 10, 1, 32, torch.float32, True, 1.0),
    (385, 10, 2, 32, torch.bfloat16, True, 1.0),
    (257, 16, 1, 32, torch.float32, False, 2.0),
    (131, 17, 1, 32, torch.float32, True, 1.0),
    (130, 1, 2, 64, torch.float32, True, 1.0),
    (4100, 1, 1, 32, torch.bfloat16, True, 1.0),
    (1031, 4, 1, 32, torch.float32, True, 1.0),
    # strips of the forward: of two rows at 2 and 4 tokens (and 10, above, in bf16), of three at 6 and 7
    (3, 2, 3, 64, torch.float32, True, 1.0),
    (3, 4, 3, 64, torch.bfloat16, True, 1.0),
    (2, 6, 3, 64, torch.float32, True, 1.0),
    (2, 7, 3, 64, torch.bfloat16, True, 1.0),
]


@pytest.mark.parametrize("B,T,H,D,dtype,bias,mult", PRODUCER_CASES)
def test_producer_parity(B, T, H, D, dtype, bias, mult):
    from mlx_vit_amd import producer_backward, producer_forward
    acts, params, cots = _prod_inputs(B, T, H, D, dtype, seed=B * 1000 + T, bias=bias)
    case = f"producer B={B} T={T} H={H} D={D} {dtype} bias={bias} mult={mult}"
    print(case, flush=True)
    da = {n: t.to(DEV) for n, t in acts.items()}
    dp = {n: (None if t is None else t.to(DEV)) for n, t in params.items()}
    dc = {n: t.to(DEV) for n, t in cots.items()}
    outs = producer_forward(da["qkv"], da["xf"], da["xb"], dp["conv_w"], dp["conv_b"], dp["dt_bias"],
                            dp["A_log"], H, D, D ** -0.5, mult, torch.float32)
    grads = producer_backward(da["qkv"], da["xf"], da["xb"], dp["conv_w"], dp["conv_b"], dp["dt_bias"],
                              dp["A_log"], dc["dq"], dc["dk"], dc["dv"], dc["dg"], dc["dbeta"], H, D, D ** -0.5,
                              mult)
    torch.cuda.synchronize()
    ref_outs, ref_grads = _prod_reference(acts, params, cots, H, D, mult)
    errs = {n: _rel(o, r) for n, o, r in zip(("q", "k", "v", "g", "beta"), outs, ref_outs)}
    names = ("qkv", "xf", "xb", "conv_w", "conv_b", "dt_bias", "A_log")
    for n, gr in zip(names, grads):
        if n == "conv_b" and not bias:
            assert gr is None
            continue
        errs["d" + n] = _rel(gr, ref_grads[n])
    _check(errs, TOL[dtype], case)


def test_producer_strided_rows():
    """q/k/v read from column slices of a wider fused projection output."""
    from mlx_vit_amd import producer_forward
    B, T, H, D = 2, 50, 4, 32
    HD = H * D
    acts, params, _ = _prod_inputs(B, T, H, D, torch.float32, seed=7)
    wide = torch.randn(B, T, 3 * HD + 64)
    wide[..., 32:32 + 3 * HD] = acts["qkv"]
    d = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    out_wide = producer_forward(d(wide)[..., 32:32 + 3 * HD], d(acts["xf"]), d(acts["xb"]), d(params["conv_w"]),
                                d(params["conv_b"]), d(params["dt_bias"]), d(params["A_log"]), H, D, 0.5)
    out_ref = producer_forward(d(acts["qkv"]), d(acts["xf"]), d(acts["xb"]), d(params["conv_w"]),
                               d(params["conv_b"]), d(params["dt_bias"]), d(params["A_log"]), H, D, 0.5)
    for a, b in zip(out_wide, out_ref):
        assert torch.equal(a, b)


def test_producer_full_size_properties():
    """Config-2 shape in bf16 (B=8, T=1568, H=12, D=64): every q row has norm
    D^-1/2 and every k row norm 1 (to bf16 rounding), g <= 0, 0 < beta < 1,
    and the forward matches the fp32 torch restatement on the GPU."""
    from mlx_vit_amd import producer_forward
    B, T, H, D = 8, 1568, 12, 64
    acts, params, _ = _prod_inputs(B, T, H, D, torch.bfloat16, seed=11)
    da = {n: t.to(DEV) for n, t in acts.items()}
    dp = {n: t.to(DEV) for n, t in params.items()}
    q, k, v, g, beta = producer_forward(da["qkv"], da["xf"], da["xb"], dp["conv_w"], dp["conv_b"], dp["dt_bias"],
                                        dp["A_log"], H, D, D ** -0.5)
    qn = q.float().reshape(B, T, -1).norm(dim=-1)
    kn = k.float().reshape(B, T, -1).norm(dim=-1)
    assert torch.allclose(qn, torch.full_like(qn, D ** -0.5), rtol=4e-3)
    assert torch.allclose(kn, torch.ones_like(kn), rtol=4e-3)
    assert bool((g <= 0).all()) and bool((beta > 0).all()) and bool((beta < 1).all())
    HD = H * D
    xq, xk, xv = da["qkv"].float().split(HD, -1)
    ref = LR.producer_from_projections(xq, xk, xv, da["xf"].float(), da["xb"].float(), dp["conv_w"],
                                       dp["conv_b"], dp["dt_bias"], dp["A_log"], H, D)
    errs = {n: _rel(o.float(), r) for n, o, r in zip(("q", "k", "v", "g", "beta"), (q, k, v, g, beta), ref)}
    _check(errs, TOL[torch.bfloat16], "producer full size")


NORM_CASES = [
    (2, 37, 3, 64, torch.float32),
    (1, 100, 12, 64, torch.float32),
    (2, 5, 4, 32, torch.float32),
    (1, 9, 16, 128, torch.float32),
    (1, 130, 2, 4, torch.float32),
    (4, 65, 12, 64, torch.bfloat16),
    (2, 37, 8, 96, torch.float32),     # D = 96: 32-lane head groups, 24 live lanes each
    (1, 20, 5, 96, torch.float32),     # an odd head count: half of the last wave idle
    (2, 30, 16, 96, torch.bfloat16),   # 16 heads of 96: eight waves
]


@pytest.mark.parametrize("B,T,H,D,dtype", NORM_CASES)
def test_gated_rmsnorm_parity(B, T, H, D, dtype):
    from mlx_vit_amd import gated_rmsnorm_backward, gated_rmsnorm_forward
    case = f"gated_rmsnorm B={B} T={T} H={H} D={D} {dtype}"
    print(case, flush=True)
    g = torch.Generator().manual_seed(T + D)
    o = torch.randn(B, T, H, D, generator=g).to(dtype)
    wide = torch.randn(B, T, H * D + 8, generator=g).to(dtype)   # the gate as a strided column slice
    w = 1 + 0.1 * torch.randn(D, generator=g)
    dy = torch.randn(B, T, H * D, generator=g).to(dtype)
    z = wide[..., 8:]
    y = gated_rmsnorm_forward(o.to(DEV), wide.to(DEV)[..., 8:], w.to(DEV), 1e-5)
    do, dz, dw = gated_rmsnorm_backward(o.to(DEV), wide.to(DEV)[..., 8:], w.to(DEV), 1e-5, dy.to(DEV))
    torch.cuda.synchronize()
    lo, lz, lw = (t.double().requires_grad_() for t in (o, z, w))
    ref = LR.gated_rms_norm(lo, lw, lz.reshape(B, T, H, D), 1e-5).reshape(B, T, H * D)
    (ref * dy.double()).sum().backward()
    errs = {"y": _rel(y, ref), "do": _rel(do, lo.grad), "dz": _rel(dz, lz.grad), "dw": _rel(dw, lw.grad)}
    _check(errs, TOL[dtype], case)


GATED_CASES = [
    # B, T, H, D, dtype, with_state, train, gate column offset (a strided gate)
    (2, 100, 3, 64, torch.bfloat16, True, False, 8),     # ragged last chunk
    (1, 1, 4, 64, torch.bfloat16, False, True, 0),       # T = 1
    (3, 64, 2, 64, torch.bfloat16, False, True, 8),      # one whole chunk
    (2, 200, 12, 64, torch.bfloat16, True, True, 0),     # four chunks (the LDS sets wrap)
    (2, 100, 3, 64, torch.float32, True, True, 4),
    (1, 77, 2, 32, torch.float32, False, False, 0),
    (2, 129, 3, 32, torch.float32, True, True, 4),       # a last chunk of one row, a strided gate
    (2, 65, 2, 64, torch.float32, False, False, 0),
    # short sequences, one wave each with its epilogue: rows for 8 and 16 tokens
    (2, 8, 3, 64, torch.bfloat16, True, True, 8),
    (87, 9, 3, 64, torch.bfloat16, True, False, 8),      # (above 256 of them at 9 to 16 tokens)
    (87, 16, 3, 64, torch.bfloat16, False, True, 0),
    (2, 7, 3, 32, torch.float32, True, True, 4),
    (2, 16, 3, 32, torch.float32, False, True, 0),
    (3, 8, 2, 64, torch.float32, False, False, 0),
    (2, 13, 2, 64, torch.float32, True, True, 4),
]


@pytest.mark.parametrize("B,T,H,D,dtype,with_state,train,pad", GATED_CASES)
def test_fwd_gated_parity(B, T, H, D, dtype, with_state, train, pad):
    """kda_fwd_gated: y against the fp64 C oracle's o followed by the fp64
    gated RMSNorm; o and the final state bit-identical to the unfused forward
    (kda_fwd / kda_fwd_train); y against the standalone norm kernel on that o;
    with the training pass, kda_bwd_train on its workspace bit-identical to the
    unfused training pair."""
    from oracle import cref
    from mlx_vit_amd import (gated_rmsnorm_forward, kda_backward_train, kda_forward, kda_forward_gated,
                             kda_forward_train)
    case = f"fwd_gated B={B} T={T} H={H} D={D} {dtype} state={with_state} train={train} pad={pad}"
    print(case, flush=True)
    x = R.make_inputs(B, T, H, D, dtype=dtype, seed=T + D, with_state=with_state, with_grad=True)
    gen = torch.Generator().manual_seed(11)
    wide = torch.randn(B, T, H * D + pad, generator=gen).to(dtype)
    w = 1 + 0.1 * torch.randn(D, generator=gen)
    d = {n: (None if t is None else t.to(DEV)) for n, t in x.items()}
    args = (d["q"], d["k"], d["v"], d["g"], d["beta"], d["s0"])
    wd = wide.to(DEV)
    y, o, sf, ws = kda_forward_gated(*args, wd[..., pad:], w.to(DEV), 1e-5, train=train)
    if train:
        o_u, sf_u, ws_u = kda_forward_train(*args)
    else:
        o_u, sf_u = kda_forward(*args)
    y_u = gated_rmsnorm_forward(o_u, wd[..., pad:], w.to(DEV), 1e-5)
    torch.cuda.synchronize()
    assert torch.equal(o, o_u), f"{case}: o differs from the unfused forward"
    assert torch.equal(sf, sf_u), f"{case}: final state differs from the unfused forward"
    ref_o = cref.forward(x["q"], x["k"], x["v"], x["g"], x["beta"], x["s0"])["o"]
    z = wide[..., pad:].double().reshape(B, T, H, D)
    ref = LR.gated_rms_norm(ref_o, w.double(), z, 1e-5).reshape(B, T, H * D)
    errs = {"y": _rel(y, ref), "y_vs_standalone": _rel(y, y_u)}
    if train:
        g1 = kda_backward_train(*args, d["do"], None, ws)
        g2 = kda_backward_train(*args, d["do"], None, ws_u)
        torch.cuda.synchronize()
        for n, a, b in zip(("dq", "dk", "dv", "dg", "dbeta", "ds0"), g1, g2):
            assert torch.equal(a, b), f"{case}: {n} from the gated forward's workspace differs"
    _check(errs, TOL[dtype], case)
    assert errs["y_vs_standalone"] <= (2e-3 if dtype == torch.bfloat16 else 1e-6), case


def test_fwd_gated_rejects():
    """Unsupported head sizes and bad gate strides raise ValueError."""
    from mlx_vit_amd import kda_forward_gated
    x = R.make_inputs(1, 10, 2, 32, dtype=torch.bfloat16, seed=1)
    d = {n: (None if t is None else t.to(DEV)) for n, t in x.items()}
    z = torch.randn(1, 10, 64, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="no fused kernel"):
        kda_forward_gated(d["q"], d["k"], d["v"], d["g"], d["beta"], None, z, torch.ones(32, device=DEV), 1e-5)
    x = R.make_inputs(1, 10, 2, 64, dtype=torch.bfloat16, seed=1)
    d = {n: (None if t is None else t.to(DEV)) for n, t in x.items()}
    with pytest.raises(ValueError, match="gate shape"):
        kda_forward_gated(d["q"], d["k"], d["v"], d["g"], d["beta"], None, z, torch.ones(64, device=DEV), 1e-5)


def _layer_params(layer):
    return {n: p.detach().cpu().double() for n, p in layer.named_parameters()}


@pytest.mark.parametrize("dtype,with_state,D,fused", [
    (torch.float32, False, 32, True), (torch.float32, True, 32, True), (torch.bfloat16, False, 32, True),
    (torch.float32, True, 64, True), (torch.float32, True, 64, False), (torch.bfloat16, True, 64, True),
    (torch.bfloat16, True, 64, False)])
def test_layer_parity(dtype, with_state, D, fused):
    """The whole GatedDeltaLayer (projections, producer, HIP recurrence, gated
    RMSNorm, o_proj) forward and backward against the fp64 restatement with
    the step recurrence (nope_gdn_mlx.py:775-885 on the 'compiled' path), with
    the output norm fused into the recurrence's store where a kernel has it
    (fused) or as the standalone kernel."""
    _layer_case(dtype, with_state, D, fused, B=2, L=100, H=3, hidden=3 * D)


@pytest.mark.parametrize("dtype,with_state", [(torch.float32, True), (torch.bfloat16, True),
                                              (torch.bfloat16, False)])
def test_layer_parity_ssv2_d96(dtype, with_state):
    """The reference's SSv2 layer, GatedDeltaLayer(768, 8, 96)
    (train_mlx_ssv2.py:71-80): head dimension 96 through the padded recurrence
    and the norm's 32-lane head groups."""
    _layer_case(dtype, with_state, 96, False, B=2, L=100, H=8, hidden=768)


def test_layer_training_step_ssv2_d96():
    """A training step of GatedDeltaLayer(768, 8, 96) in bf16: forward,
    backward, AdamW update; every parameter gets a finite, nonzero gradient,
    the update changes the parameters, and the loss of the next forward on the
    same batch is lower."""
    from mlx_vit_amd import GatedDeltaLayer
    torch.manual_seed(5)
    layer = GatedDeltaLayer(768, 8, 96).to(torch.bfloat16)
    layer.A_log.data = layer.A_log.data.float()
    layer.dt_bias.data = layer.dt_bias.data.float()
    layer = layer.to(DEV)
    g = torch.Generator().manual_seed(6)
    x = torch.randn(2, 1568, 768, generator=g).to(torch.bfloat16).to(DEV)
    target = torch.randn(2, 1568, 768, generator=g).to(torch.bfloat16).to(DEV)
    # lr 1e-2: an AdamW step of about lr moves even a bf16 weight at 1.0 (spacing 2^-7)
    opt = torch.optim.AdamW(layer.parameters(), lr=1e-2)
    before = {n: p.detach().clone() for n, p in layer.named_parameters()}
    losses = []
    for _ in range(2):
        out, _ = layer(x)
        loss = ((out.float() - target.float()) ** 2).mean()
        opt.zero_grad()
        loss.backward()
        if not losses:
            for n, p in layer.named_parameters():
                assert p.grad is not None and torch.isfinite(p.grad).all() and p.grad.abs().sum() > 0, n
        opt.step()
        losses.append(loss.item())
    torch.cuda.synchronize()
    print("ssv2 layer training step losses", losses, flush=True)
    assert losses[1] < losses[0]
    assert all(not torch.equal(before[n], p.detach()) for n, p in layer.named_parameters())


def _layer_case(dtype, with_state, D, fused, B, L, H, hidden):
    from mlx_vit_amd import GatedDeltaLayer
    case = f"layer B={B} L={L} hidden={hidden} H={H} D={D} {dtype} state={with_state} fused={fused}"
    print(case, flush=True)
    torch.manual_seed(3)
    layer = GatedDeltaLayer(hidden, H, D)
    layer.fused_output_norm = fused
    with torch.no_grad():
        layer.dt_bias.normal_(0, 0.1)
        layer.o_norm.weight.normal_(1, 0.1)
    layer = layer.to(dtype)
    # A_log and dt_bias stay fp32 in a bf16 model (nope_gdn_mlx.py:4959-4963)
    layer.A_log.data = layer.A_log.data.float()
    layer.dt_bias.data = layer.dt_bias.data.float()
    g = torch.Generator().manual_seed(4)
    x = torch.randn(B, L, hidden, generator=g).to(dtype)
    s0 = 0.1 * torch.randn(B, H, D, D, generator=g) if with_state else None
    cot = torch.randn(B, L, hidden, generator=g).to(dtype)
    cot_s = torch.randn(B, H, D, D, generator=g)
    ref_params = _layer_params(layer)
    layer = layer.to(DEV)
    xd = x.to(DEV).requires_grad_()
    s0d = None if s0 is None else s0.to(DEV).requires_grad_()
    out, st = layer(xd, s0d)
    ((out.float() * cot.to(DEV).float()).sum() + (st * cot_s.to(DEV)).sum()).backward()
    torch.cuda.synchronize()

    rp = {n: t.requires_grad_() for n, t in ref_params.items()}
    rx = x.double().requires_grad_()
    rs0 = None if s0 is None else s0.double().requires_grad_()
    keep = {}
    rout, rst = LR.layer_forward(rp, rx, H, D, rs0, keep=keep)
    keep["g"].retain_grad()
    ((rout * cot.double()).sum() + (rst * cot_s.double()).sum()).backward()
    errs = {"out": _rel(out, rout), "state": _rel(st, rst), "dx": _rel(xd.grad, rx.grad)}
    if s0 is not None:
        errs["ds0"] = _rel(s0d.grad, rs0.grad)
    for n, p in layer.named_parameters():
        errs["d" + n] = _rel(p.grad, rp[n].grad)
    # dA_log[h] is the signed sum over (b, t, d) of dg * g (dg/dA_log = g): its
    # error is bounded relative to the sum of the terms' magnitudes, which
    # cancellation can make far larger than the sum itself (the rel-L2 of an
    # H-entry vector of such sums is printed, not asserted)
    terms = (keep["g"].grad * keep["g"]).abs().sum(dim=(0, 1, 3))
    plain = errs.pop("dA_log")
    errs["dA_log/sum|terms|"] = (layer.A_log.grad.detach().cpu().double() - rp["A_log"].grad).norm().item() / \
        terms.norm().item()
    print(case, f"dA_log rel-L2 {plain:.2e}, cancellation factor {terms.norm().item() / rp['A_log'].grad.norm().item():.1f}",
          flush=True)
    _check(errs, TOL[dtype], case)


@pytest.mark.parametrize("B,T,H,D,dtype,with_state,shift", [
    (2, 100, 3, 64, torch.float32, True, 1.5),
    (1, 130, 2, 32, torch.float32, False, 1.5),
    (2, 77, 4, 64, torch.bfloat16, True, 1.5),       # bf16 D <= 64: one decay per (b, t, h) in the kernels
    (1, 150, 2, 32, torch.bfloat16, False, 1.5),
    (1, 130, 2, 64, torch.bfloat16, True, -4.0),     # alpha down to ~0.002: beyond the span guard
])
def test_chunk_gdn_parity(B, T, H, D, dtype, with_state, shift):
    """Scalar-alpha GDN (the reference's original gated delta rule) through the
    KDA kernels against the fp64 step loop (nope_gdn_mlx.py:641-650, 919-947):
    outputs and the gradients of q, k, v, alpha, beta and the initial state."""
    from mlx_vit_amd import chunk_gdn
    case = f"chunk_gdn B={B} T={T} H={H} D={D} {dtype} state={with_state} shift={shift}"
    print(case, flush=True)
    g = torch.Generator().manual_seed(T + D)
    x = R.make_inputs(B, T, H, D, dtype=dtype, seed=T, with_state=with_state, with_grad=True)
    alpha = torch.sigmoid(torch.randn(B, T, H, generator=g) + shift)   # shift 1.5: 0.2 .. 0.98
    cot_s = torch.randn(B, H, D, D, generator=g)
    dev = {n: x[n].to(DEV).requires_grad_() for n in ("q", "k", "v", "beta")}
    a_d = alpha.to(DEV).requires_grad_()
    s0_d = None if x["s0"] is None else x["s0"].to(DEV).requires_grad_()
    o, st = chunk_gdn(dev["q"], dev["k"], dev["v"], a_d, dev["beta"], s0_d)
    ((o.float() * x["do"].to(DEV).float()).sum() + (st * cot_s.to(DEV)).sum()).backward()
    torch.cuda.synchronize()
    ref = {n: x[n].double().requires_grad_() for n in ("q", "k", "v", "beta")}
    a_r = alpha.double().requires_grad_()
    s0_r = None if x["s0"] is None else x["s0"].double().requires_grad_()
    ro, rst = R.loop_compiled_gdn(ref["q"], ref["k"], ref["v"], a_r, ref["beta"], s0_r, compute_dtype=torch.float64)
    ((ro * x["do"].double()).sum() + (rst * cot_s.double()).sum()).backward()
    errs = {"o": _rel(o, ro), "state": _rel(st, rst), "dalpha": _rel(a_d.grad, a_r.grad)}
    for n in ("q", "k", "v", "beta"):
        errs["d" + n] = _rel(dev[n].grad, ref[n].grad)
    if s0_d is not None:
        errs["ds0"] = _rel(s0_d.grad, s0_r.grad)
    _check(errs, TOL[dtype], case)


def test_layer_parity_scalar_alpha():
    """GatedDeltaLayer(channel_wise_decay=False): a_proj gate, producer without
    the decay gate, path hip_chunkwise_gdn, against the fp64 restatement."""
    from mlx_vit_amd import GatedDeltaLayer
    B, L, hidden, H, D = 2, 90, 64, 2, 32
    torch.manual_seed(5)
    layer = GatedDeltaLayer(hidden, H, D, channel_wise_decay=False)
    g = torch.Generator().manual_seed(6)
    x = torch.randn(B, L, hidden, generator=g)
    cot = torch.randn(B, L, hidden, generator=g)
    cot_s = torch.randn(B, H, D, D, generator=g)
    ref_params = _layer_params(layer)
    layer = layer.to(DEV)
    xd = x.to(DEV).requires_grad_()
    out, st = layer(xd)
    ((out * cot.to(DEV)).sum() + (st * cot_s.to(DEV)).sum()).backward()
    torch.cuda.synchronize()
    rp = {n: t.requires_grad_() for n, t in ref_params.items()}
    rx = x.double().requires_grad_()
    rout, rst = LR.layer_forward(rp, rx, H, D)
    ((rout * cot.double()).sum() + (rst * cot_s.double()).sum()).backward()
    errs = {"out": _rel(out, rout), "state": _rel(st, rst), "dx": _rel(xd.grad, rx.grad)}
    for n, p in layer.named_parameters():
        errs["d" + n] = _rel(p.grad, rp[n].grad)
    _check(errs, TOL[torch.float32], "layer scalar alpha")


@pytest.mark.parametrize("rows,shapes", [
    (1, [(8, 8, True)]), (31, [(12, 64, True)]), (33, [(64, 72, False), (12, 8, True)]),
    (224, [(130, 192, True)]), (257, [(128, 128, False), (200, 64, True), (300, 136, True)]),
    (3000, [(140, 128, True), (64, 256, False)])])
def test_weight_grads_parity(rows, shapes):
    """weight_grads against the fp32 products: one and several problems, tails of
    the 32-row steps, of the 128 and 64 wide tiles and of the row splits (one
    split below 512 rows).  fp32 sums of bf16 operands rounded once: 2^-8 an
    element at most.  dy as a column slice of a wider matrix."""
    from mlx_vit_amd.layer import weight_grads
    gen = torch.Generator().manual_seed(rows)
    probs = []
    for n, k, bias in shapes:
        wide = torch.randn(rows, -(-n // 8) * 8 + 16, generator=gen).to(torch.bfloat16).to(DEV)
        probs.append((wide[:, 8:8 + n], torch.randn(rows, k, generator=gen).to(torch.bfloat16).to(DEV), bias))
    got = weight_grads(probs, rows)
    torch.cuda.synchronize()
    for (dy, x, bias), (dw, db) in zip(probs, got):
        ref = {"dw": dy.double().cpu().T @ x.double().cpu(), "db": dy.double().cpu().sum(0)}
        errs = {"dw": _rel(dw, ref["dw"])}
        if bias:
            errs["db"] = _rel(db, ref["db"])
        _check(errs, 2.0 ** -8, f"weight_grads rows={rows} n={dy.shape[1]} k={x.shape[1]}")


@pytest.mark.parametrize("H,D,L,frozen,contiguous", [(3, 64, 100, False, True), (2, 32, 8, True, True),
                                                     (8, 96, 70, False, False)])
def test_layer_one_node_matches_modules(H, D, L, frozen, contiguous):
    """The layer as one autograd node against the same layer run module by module
    (a forward hook on one of its maps sends it there, and is called): outputs
    and every gradient to the bf16 bar, with a state, frozen parameters, a
    non-contiguous input, and with only the new state used."""
    from mlx_vit_amd import GatedDeltaLayer
    from mlx_vit_amd.layer_fused import fused_params
    from mlx_vit_amd.model import to_bf16
    torch.manual_seed(7)
    layer = to_bf16(GatedDeltaLayer(H * D, H, D)).to(DEV)
    if frozen:
        for n, p in layer.named_parameters():
            p.requires_grad_(n.startswith("g_proj") or n == "A_log" or n == "k_conv1d.weight")
    gen = torch.Generator().manual_seed(L)
    x = torch.randn(2, L, H * D, generator=gen).to(torch.bfloat16).to(DEV)
    if not contiguous:
        x = x.transpose(0, 1).contiguous().transpose(0, 1)
    s0 = (0.1 * torch.randn(2, H, D, D, generator=gen)).to(DEV).requires_grad_()
    dout = torch.randn(2, L, H * D, generator=gen).to(torch.bfloat16).to(DEV)
    ds = torch.randn(2, H, D, D, generator=gen).to(DEV)
    x.requires_grad_()
    leaves = [("x", x), ("s0", s0)] + [(n, p) for n, p in layer.named_parameters() if p.requires_grad]

    def grads(outs, cots):
        got = torch.autograd.grad(outs, [t for _, t in leaves], cots, allow_unused=True)
        return {n: g for (n, _), g in zip(leaves, got) if g is not None}

    assert fused_params(layer, x, s0) is not None
    out, s = layer(x, s0)
    one = grads([out, s], [dout, ds])
    only_state = grads([layer(x, s0)[1]], [ds])
    with torch.no_grad():
        out_ng, s_ng = layer(x, s0)
    calls = []
    handle = layer.b_proj.register_forward_hook(lambda *a: calls.append(1))
    assert fused_params(layer, x, s0) is None
    out_m, s_m = layer(x, s0)
    mods = grads([out_m, s_m], [dout, ds])
    mods_state = grads([layer(x, s0)[1]], [ds])
    handle.remove()
    torch.cuda.synchronize()
    assert len(calls) == 2 and set(one) == set(mods) and set(only_state) == set(mods_state)
    errs = {"out": _rel(out, out_m), "s": _rel(s, s_m), "out_ng": _rel(out_ng, out_m), "s_ng": _rel(s_ng, s_m)}
    errs.update({n: _rel(g, mods[n]) for n, g in one.items()})
    # (the maps behind the output get no gradient here, q and its conv zeros)
    errs.update({"state:" + n: _rel(g, mods_state[n]) if mods_state[n].abs().max() > 0 else g.abs().max().item()
                 for n, g in only_state.items()})
    for n, g in one.items():
        assert g.dtype == mods[n].dtype and g.shape == mods[n].shape, n
    _check(errs, 1e-2, f"one node H={H} D={D} L={L}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 255, 1000])
def test_log_decay(n, dtype):
    """The scalar decay's logarithm and its adjoint against torch's clamp(log) on
    the same values, alpha = 0, the clamp's edge and alpha = 1 among them, and a
    strided alpha: g to one fp32 rounding of the logarithm, d alpha to alpha's
    own rounding."""
    from mlx_vit_amd.kda import GDN_LOG_ALPHA_MIN, _log_alpha
    gen = torch.Generator().manual_seed(n)
    a = torch.rand(2 * n, generator=gen)
    a[:8] = torch.tensor([0.0, 1.0, 0.5, 1e-38, 1e-30, 0.999, 1e-35, 1e-34])[:min(8, 2 * n)]
    al = a.to(dtype).to(DEV)[::2].requires_grad_()
    ref = al.detach().clone().requires_grad_()
    dg = torch.randn(n, generator=gen).to(DEV)
    g = _log_alpha(al)
    (da,) = torch.autograd.grad(g, al, dg)
    gr = torch.clamp(torch.log(ref.float()), min=GDN_LOG_ALPHA_MIN)
    (dr,) = torch.autograd.grad(gr, ref, dg)
    torch.cuda.synchronize()
    assert torch.allclose(g, gr, rtol=2.0 ** -22, atol=2.0 ** -23)
    fin = torch.isfinite(dr.float())
    assert torch.equal(fin, torch.isfinite(da.float()))
    assert torch.allclose(da.float()[fin], dr.float()[fin], rtol=2.0 ** (-8 if dtype == torch.bfloat16 else -22), atol=0.0)


def _bf16_layer(H, D, seed=7):
    from mlx_vit_amd import GatedDeltaLayer
    from mlx_vit_amd.model import to_bf16
    torch.manual_seed(seed)
    return to_bf16(GatedDeltaLayer(H * D, H, D)).to(DEV)


def _bf16_randn(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).to(DEV)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.filterwarnings("ignore")
def test_layer_jit_trace(grad):
    """A traced bf16 layer computes what the layer does, on other inputs than
    those it was traced with (the same kernels: the same bits)."""
    layer = _bf16_layer(3, 64).requires_grad_(grad)
    x, y = _bf16_randn(1, 2, 100, 192), _bf16_randn(2, 2, 100, 192)
    with torch.set_grad_enabled(grad):
        traced = torch.jit.trace(layer, (x,), check_trace=False)
        got = traced(y)
        handle = layer.b_proj.register_forward_hook(lambda *a: None)   # module by module, as traced
        ref = layer(y)
        handle.remove()
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


def test_layer_refuses_forward_mode():
    """The kernels have no forward-mode derivative: a tangent on x, or on a weight,
    is refused, with or without gradients, and never dropped."""
    from torch.autograd import forward_ad
    layer = _bf16_layer(3, 64)
    x = _bf16_randn(1, 2, 20, 192)
    for trained in (True, False):
        layer.requires_grad_(trained)
        with forward_ad.dual_level(), pytest.raises(NotImplementedError):
            layer(forward_ad.make_dual(x, torch.ones_like(x)))
        with forward_ad.dual_level(), pytest.raises(NotImplementedError):
            w = layer.q_proj.weight.detach()
            dual = forward_ad.make_dual(w, torch.ones_like(w))
            torch.func.functional_call(layer, {"q_proj.weight": dual}, (x,))
        layer(x)


@pytest.mark.parametrize("H,D,L", [(3, 64, 100), (2, 64, 8), (8, 96, 70)])
def test_layer_second_backward(H, D, L):
    """Two backwards over one retained graph: the first uses the training forward's
    workspace, the second forms the factors again, the same bits; and the output's
    and the state's gradients taken apart add up to the joint ones."""
    layer = _bf16_layer(H, D)
    x = _bf16_randn(1, 2, L, H * D).requires_grad_()
    s0 = (0.1 * _bf16_randn(2, 2, H, D, D).float()).requires_grad_()
    dout, ds = _bf16_randn(3, 2, L, H * D), _bf16_randn(4, 2, H, D, D).float()
    leaves = [x, s0, *layer.parameters()]
    out, s = layer(x, s0)

    def grads(outs, cots):
        return torch.autograd.grad(outs, leaves, cots, retain_graph=True, allow_unused=True)

    first, second = grads([out, s], [dout, ds]), grads([out, s], [dout, ds])
    parts = list(zip(grads([out], [dout]), grads([s], [ds])))
    torch.cuda.synchronize()
    for a, b in zip(first, second):
        assert torch.equal(a, b)
    _check({str(i): _rel(a.float() + (0 if b is None else b.float()), t)
            for i, ((a, b), t) in enumerate(zip(parts, first))}, TOL[torch.bfloat16], f"second backward {H} {D} {L}")


@pytest.mark.parametrize("offset", [1, 4])
def test_layer_unaligned_inputs(offset):
    """x and the output's cotangent at a storage offset that is no multiple of 16
    bytes: the same bits as from aligned copies, gradients included."""
    layer = _bf16_layer(3, 64)

    def shifted(t):
        return torch.empty(t.numel() + offset, dtype=t.dtype, device=DEV)[offset:].view_as(t).copy_(t)

    def run(x, dout):
        x = x.requires_grad_()
        out, s = layer(x)
        return [out, s, *torch.autograd.grad(out, [x, *layer.parameters()], dout)]

    x, dout = _bf16_randn(1, 2, 50, 192), _bf16_randn(2, 2, 50, 192)
    ref, got = run(x, dout), run(shifted(x.detach()), shifted(dout))
    assert shifted(dout).data_ptr() % 16 != 0 and shifted(dout).is_contiguous()
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n,k,ld,offset", [(12, 8, 13, 0), (8, 16, 24, 3), (20, 24, 24, 8)])
def test_weight_grads_any_rows(n, k, ld, offset):
    """Rows that the kernel cannot read 16 bytes at a time -- odd strides, bases and
    widths -- are copied: the same bits as from aligned operands."""
    from mlx_vit_amd.layer import weight_grads
    rows, wide = 40, max(ld, n) + offset
    dy = _bf16_randn(n, rows, wide)[:, offset:offset + n]
    x = _bf16_randn(k, rows, k + ld)[:, 1:1 + k]
    ref = torch.empty(rows, -(-n // 8) * 8, dtype=torch.bfloat16, device=DEV)[:, :n].copy_(dy)
    (dw, db), (rw, rb) = weight_grads([(dy, x, True)], rows) + weight_grads([(ref, x.contiguous(), True)], rows)
    assert torch.equal(dw, rw) and torch.equal(db, rb)


def test_layer_output_in_place():
    """The layer's outputs take in-place operations: under autograd, and a result
    formed without gradients that later enters a graph."""
    layer = _bf16_layer(3, 64)
    x, dout = _bf16_randn(1, 2, 20, 192), _bf16_randn(2, 2, 20, 192)
    out, s = layer(x)
    ref = torch.autograd.grad([2 * out, s], list(layer.parameters()), [dout, torch.ones_like(s)])
    out, s = layer(x)
    with torch.no_grad():
        plain, _ = layer(x)
    out *= 2
    s += 1
    for a, b in zip(torch.autograd.grad([out, s], list(layer.parameters()), [dout, torch.ones_like(s)]), ref):
        assert torch.equal(a, b)
    plain += torch.ones(1, dtype=plain.dtype, device=DEV, requires_grad=True)
    assert plain.requires_grad and torch.equal(plain, 1 + out / 2)


def _records(fn):
    """(fn(), the ids of the library's kernels that it launched)."""
    from mlx_vit_amd import _lib
    import ctypes
    lib = _lib.load()
    lib.kda_profile_enable(1)
    try:
        out = fn()
        torch.cuda.synchronize()
    finally:
        lib.kda_profile_enable(0)
    ms, n, ids = ctypes.c_double(), ctypes.c_int(), set()
    for i in range(_lib.PROF_NKERNELS):
        _lib.check(lib.kda_profile_read(i, ctypes.byref(ms), ctypes.byref(n)), "kda_profile_read")
        if n.value:
            ids.add(i)
    return out, ids


_PREP_TRAIN, _LOCAL, _PRODUCER_BWD, _NORM_BWD = 6, 5, 8, 10
_WHOLE = {_PREP_TRAIN, _LOCAL, _PRODUCER_BWD, _NORM_BWD}


@pytest.mark.parametrize("trained,backward_kernels,problems", [
    (("o_proj",), set(), [(192, 192)]),
    (("o_norm",), {_NORM_BWD}, []),
    (("g_proj_2.bias",), {_NORM_BWD}, [(192, 64)]),
    (("g_proj_1", "o_proj"), {_NORM_BWD}, [(64, 192), (192, 192)]),
    (("k_proj",), _WHOLE, [(576, 192)]),
    (("q_proj", "f_proj_1"), _WHOLE, [(640, 192)]),
    (("f_proj_1", "b_proj"), _WHOLE, [(64, 192), (3, 192)]),
    (("f_proj_2", "v_conv1d"), _WHOLE, [(192, 64)]),
    (("A_log", "dt_bias"), _WHOLE, []),
    (("x",), _WHOLE, []),
    (("state",), _WHOLE - {_PRODUCER_BWD}, []),
])
def test_layer_frozen_parameters(trained, backward_kernels, problems, monkeypatch):
    """With some parameters frozen the layer launches what their gradients need and
    no more -- recurrence, producer and norm backward, weight gradients by shape
    -- and those gradients are the ones of the layer trained whole (the sums over
    the tokens in another split: bf16 results by their own rounding)."""
    from mlx_vit_amd import layer as layer_module
    H, D, L = 3, 64, 100
    layer = _bf16_layer(H, D)
    x, s0 = _bf16_randn(1, 2, L, H * D), 0.1 * _bf16_randn(2, 2, H, D, D).float()
    dout = _bf16_randn(3, 2, L, H * D)
    shapes = []
    weight_grads = layer_module.weight_grads
    monkeypatch.setattr(layer_module, "weight_grads", lambda p, rows: (
        shapes.extend((dy.shape[1], t.shape[1]) for dy, t, _ in p), weight_grads(p, rows))[1])

    def run(pick):
        named = [("x", x.detach()), ("state", s0.detach()), *layer.named_parameters()]
        leaves = {n: t.requires_grad_(pick(n)) for n, t in named if t.is_leaf}
        out, s = layer(leaves["x"], leaves["state"])
        want = [n for n in leaves if pick(n)]
        return out, s, dict(zip(want, torch.autograd.grad(out, [leaves[n] for n in want], dout)))

    out, s, ref = run(lambda n: True)
    shapes.clear()
    (out_f, s_f, got), ids = _records(lambda: run(lambda n: n.startswith(trained)))
    assert ids & _WHOLE == backward_kernels and sorted(shapes) == sorted(problems)
    through = bool(backward_kernels & {_LOCAL})
    assert out_f.requires_grad and s_f.requires_grad == through
    assert torch.equal(out, out_f) and torch.equal(s, s_f)
    _check({n: _rel(g, ref[n]) for n, g in got.items()}, TOL[torch.bfloat16], f"frozen all but {trained}")


def test_layer_create_graph():
    """Gradients taken with create_graph keep the graph that the separate modules
    give them: the same first gradients, and the same derivatives of a function of
    them (through the linear maps; the kernels' adjoints have none), to the bf16 bar
    (the cotangent 2 out comes from the one node's forward, whose products are
    stacked)."""
    layer = _bf16_layer(3, 64)
    x0, s0 = _bf16_randn(1, 2, 50, 192), 0.1 * _bf16_randn(2, 2, 3, 64, 64).float()
    names = [n for n, _ in layer.named_parameters()]

    def run():
        x = x0.clone().requires_grad_()
        leaves = [x, *layer.parameters()]
        out, s = layer(x, s0)
        first = torch.autograd.grad([out.square().sum(), s.square().sum()], leaves, create_graph=True)
        assert all(t.requires_grad for t in first[:1])
        penalty = sum(t.float().square().sum() for t in first)
        return first, torch.autograd.grad(penalty, leaves, allow_unused=True)

    first, second = run()
    handle = layer.b_proj.register_forward_hook(lambda *a: None)   # module by module
    first_m, second_m = run()
    handle.remove()
    assert [t is None for t in second] == [t is None for t in second_m]
    errs = {n: _rel(a, b) for n, a, b in zip(["x"] + names, first, first_m)}
    errs.update({"second:" + n: _rel(a, b) for n, a, b in zip(["x"] + names, second, second_m) if a is not None})
    _check(errs, TOL[torch.bfloat16], "create_graph")
    out, _ = layer(x0)
    with torch.no_grad():
        layer.q_proj.weight.mul_(1.0)
    with pytest.raises(RuntimeError, match="modified in place"):
        torch.autograd.grad(out.sum(), layer.q_proj.weight, create_graph=True)


def test_layer_inference_tensor_input():
    """x made under inference_mode with a gradient wanted for the state only: nothing
    of x has to be saved, and the layer takes it, as the separate modules do."""
    layer = _bf16_layer(3, 64).requires_grad_(False)
    plain = _bf16_randn(1, 2, 50, 192)
    with torch.inference_mode():
        x = plain.clone()
    grads = []
    for t in (x, plain):
        s0 = (0.1 * _bf16_randn(2, 2, 3, 64, 64).float()).requires_grad_()
        out, s = layer(t, s0)
        grads += [out.detach(), *torch.autograd.grad([out.float().sum(), s.sum()], s0)]
    _check({"out": _rel(grads[0], grads[2]), "ds0": _rel(grads[1], grads[3])}, TOL[torch.bfloat16], "inference x")


def test_layer_inference_memory():
    """Without gradients the layer as one node holds no more memory at a time than
    module by module (its stacked weight has the gates' rows besides q, k and v's)."""
    H, D, B, L = 4, 64, 4, 4096
    layer = _bf16_layer(H, D)
    x = _bf16_randn(1, B, L, H * D)

    def peak():
        with torch.no_grad():
            layer(x)   # the allocator's first use of these sizes
            torch.cuda.synchronize()
            torch.cuda.reset_peak_memory_stats()
            base = torch.cuda.memory_allocated()
            out = layer(x)
            torch.cuda.synchronize()
        return torch.cuda.max_memory_allocated() - base

    one = peak()
    handle = layer.b_proj.register_forward_hook(lambda *a: None)
    modules = peak()
    handle.remove()
    print("inference memory", one, modules, flush=True)
    assert one <= modules + 2 * H * D * (2 * D + H + 8) + 4096
