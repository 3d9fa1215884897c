"""Register storage in scaling form: potentials that move further than the plan entries'
bases allow (the bases move along, or the workgroup forms its entries anew), few iterations (the entries' common
shift not yet taken), and the edges of the register tiles, for the plain, the history and
the balanced forward.  Float64 oracles; normwise bar 1e-4 (fp32 inputs)."""

import math

import numpy as np
import pytest
import torch

from conftest import assert_close_rel
from oracle import balanced_transport as bt
from oracle import sinkhorn as ref

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
MAX_DRIFT = 44 * math.log(2.0)  # nats: move of a potential that the forward's entries take
MAX_FACTOR = 32 * math.log(2.0)  # nats: factor of a plan that the backwards' entries take


def _uot(B, H, N, d, K, seed, v_scale, lengths):
    g = torch.Generator().manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g)
    t = dict(Q=rn(B, H, N, d), K=rn(B, H, N, d), V=rn(B, H, N, d), G=rn(B, H, N, d), x_res=rn(B, N, 3),
             pos_weight=torch.zeros(H, 68), eps=torch.linspace(0.3, 1.0, H), w_dist=torch.zeros(H),
             log_v_init=v_scale * rn(B, H, N), log_u_init=torch.zeros(B, H, N))
    mask = torch.zeros(B, N)
    lmu, lnu = torch.zeros(B, H, N), torch.zeros(B, H, N)
    for b, n in enumerate(lengths):
        mask[b, :n] = 1
        lmu[b, :, :n] = torch.log_softmax(rn(H, n), -1)
        lnu[b, :, :n] = torch.log_softmax(rn(H, n), -1)
    t["log_v_init"] *= mask[:, None, :]
    t.update(log_mu=lmu, log_nu=lnu, mask=mask)
    return t


@pytest.mark.parametrize("unrolled", [False, True])
@pytest.mark.parametrize("B,H,N,d,K,v_scale,lengths", [
    (1, 4, 256, 32, 1, 0.5, [256]),     # the tail follows the sweeps that formed the entries
    (1, 4, 250, 32, 2, 40.0, [250]),    # initial potentials far from the first update: formed anew
    (2, 8, 300, 32, 5, 40.0, [300, 161]),
    (2, 8, 500, 24, 3, 0.5, [497, 16]),  # a member without a second tile, and one without any
    (1, 8, 200, 64, 3, 40.0, [200]),    # head dim 64: the recomputing tail
])
def test_register_forward(B, H, N, d, K, v_scale, lengths, unrolled):
    from deepfold_amd import flash_sinkhorn_attn

    print(f"case B{B} H{H} N{N} d{d} K{K} v{v_scale} unrolled={unrolled}", flush=True)
    t = _uot(B, H, N, d, K, N + K, v_scale, lengths)
    c = {k: v.to(DEV) for k, v in t.items()}
    out = flash_sinkhorn_attn(c["Q"], c["K"], c["V"], c["G"], c["x_res"], c["pos_weight"], None, c["eps"], None,
                              c["log_mu"], c["log_nu"], K_iter=K, log_u_init=c["log_u_init"],
                              log_v_init=c["log_v_init"], mask=c["mask"],
                              ift_mode="unrolled" if unrolled else "reference")
    n64 = {k: v.double().numpy() for k, v in t.items()}
    args = dict(Q=n64["Q"], K=n64["K"], V=n64["V"], G=n64["G"], x_res=n64["x_res"], pos_weight=n64["pos_weight"],
                pos_bins=None, eps=n64["eps"], w_dist=n64["w_dist"], log_mu=n64["log_mu"], log_nu=n64["log_nu"],
                log_u_init=n64["log_u_init"], log_v_init=n64["log_v_init"], mask=n64["mask"])
    want = ref.forward(K_iter=K, **args)
    if v_scale > 1:  # the case moves some potential past the bound
        one = ref.forward(K_iter=1, **args)
        assert np.max(np.abs(one["log_v"] - n64["log_v_init"])) > MAX_DRIFT
    valid = t["mask"].numpy()[:, None, :, None]
    for name, got in zip(("o_flat", "x_centroid", "log_u", "log_v"), out):
        w = want[name] * (valid if name == "x_centroid" else 1.0)
        assert_close_rel(got.detach().cpu().double().numpy(), w, 1e-4, name)


# common: every logit 160 nats up, which moves all column potentials alike in the first iteration and leaves
# their spread (the bases move along); marginals: some log nu at -70, and eps: below 0.075 (the first
# iteration runs on the logits)
@pytest.mark.parametrize("unrolled", [False, True])
@pytest.mark.parametrize("what,B,H,N,d,K", [
    ("common", 1, 4, 250, 32, 6), ("common", 1, 8, 500, 32, 2), ("common", 2, 4, 700, 24, 4), ("common", 1, 4, 200, 64, 3),
    ("marginals", 1, 4, 250, 32, 2), ("marginals", 2, 8, 390, 32, 5), ("marginals", 1, 4, 700, 32, 3),
    ("eps", 1, 4, 250, 32, 2), ("eps", 1, 8, 390, 32, 8), ("eps", 1, 4, 200, 64, 5),
])
def test_register_forward_moves(what, B, H, N, d, K, unrolled):
    from deepfold_amd import flash_sinkhorn_attn

    print(f"case {what} B{B} H{H} N{N} d{d} K{K} unrolled={unrolled}", flush=True)
    t = _uot(B, H, N, d, K, N + K, 0.0, [N] * B)
    bins = None
    if what == "common":
        t["eps"] = torch.ones(H)
        t["pos_weight"] = torch.full((H, 68), -160.0)
        bins = torch.zeros(B, N, N, dtype=torch.int32)
    elif what == "marginals":
        t["log_nu"][..., 5:8] = -70.0
    else:
        t["eps"] = torch.linspace(0.03, 0.07, H)
    n64 = {k: v.double().numpy() for k, v in t.items()}
    args = dict(Q=n64["Q"], K=n64["K"], V=n64["V"], G=n64["G"], x_res=n64["x_res"], pos_weight=n64["pos_weight"],
                pos_bins=None if bins is None else bins.numpy(), eps=n64["eps"], w_dist=n64["w_dist"],
                log_mu=n64["log_mu"], log_nu=n64["log_nu"])
    want = ref.forward(K_iter=K, **args)
    one = ref.forward(K_iter=1, **args)["log_v"]  # the first move: the potentials start at zero
    if what == "common":
        assert np.abs(one).max() > MAX_DRIFT and np.abs(one.max(-1) + one.min(-1)).max() / 2 < 64 * math.log(2.0)
        assert (one.max(-1) - one.min(-1)).max() / 2 < 34 * math.log(2.0)
    else:
        assert np.abs(one).max() > 24 * math.log(2.0)
    c = {k: v.to(DEV) for k, v in t.items()}
    out = flash_sinkhorn_attn(c["Q"], c["K"], c["V"], c["G"], c["x_res"], c["pos_weight"],
                              None if bins is None else bins.to(DEV), c["eps"], None, c["log_mu"], c["log_nu"],
                              K_iter=K, ift_mode="unrolled" if unrolled else "reference")
    # the fp32 logits: 2^-24 of their largest (230 in log2 units, 200 at eps 0.03) enters every entry
    for name, got in zip(("o_flat", "x_centroid", "log_u", "log_v"), out):
        assert_close_rel(got.detach().cpu().double().numpy(), want[name], 1e-4, name)


@pytest.mark.parametrize("B,H,N,d,K,eps,lengths", [
    (1, 16, 256, 32, 1, 0.5, None),
    (1, 8, 250, 32, 6, 0.01, None),          # logits of +-100 nats: formed anew
    (2, 16, 384, 32, 4, 0.02, [384, 200]),   # three tiles a member
    (1, 8, 130, 64, 5, 0.02, [117]),         # the recomputing tail
])
def test_register_balanced(B, H, N, d, K, eps, lengths):
    from deepfold_amd import balanced_sinkhorn_transport_dual

    print(f"case B{B} H{H} N{N} d{d} K{K} eps{eps}", flush=True)
    g = torch.Generator().manual_seed(N + K)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    Q, Kk = unit(torch.randn(B, H, N, d, generator=g)), unit(torch.randn(B, H, N, d, generator=g))
    Kk[:, :, 0] = Q[:, :, 0]  # one aligned pair: a column potential far from the others
    x, V = 3 * torch.randn(B, N, 3, generator=g), torch.randn(B, H, N, d, generator=g)
    e, al, r = torch.full((H,), eps), torch.full((H,), -1.0), torch.full((H,), 10.0)
    mask = None
    if lengths is not None:
        mask = torch.zeros(B, N)
        for b, n in enumerate(lengths):
            mask[b, :n] = 1
    dev = lambda t: None if t is None else t.to(DEV)
    xc, hc = balanced_sinkhorn_transport_dual(dev(Q), dev(Kk), dev(x), dev(V), dev(e), dev(al), dev(r), K_iter=K,
                                              mask=dev(mask))
    f = lambda t: None if t is None else t.double()
    wx, wh = bt.balanced_transport_dual(f(Q), f(Kk), f(x), f(V), f(e), f(al), f(r), K_iter=K, mask=f(mask))
    # sharp plans: the logits' fp32 rounding (2^-24 of 100 nats) enters every entry
    tol = 1e-4
    assert_close_rel(xc.cpu().double().numpy(), wx.numpy(), tol, "x_centroid")
    assert_close_rel(hc.cpu().double().numpy(), wh.numpy(), tol, "h_centroid")


@pytest.mark.parametrize("B,H,N,d,K,eps,lengths,tol", [
    (1, 8, 70, 32, 33, 1.0, None, 1e-4),          # odd iteration count, more than one batch of factors
    (1, 4, 40, 16, 64, 1.0, None, 1e-4),          # the most iterations whose vectors are kept
    (1, 4, 40, 16, 65, 1.0, None, 1e-4),          # one more: the general sweeps
    (2, 8, 300, 32, 1, 0.5, [300, 163], 1e-4),    # a single iteration: no recurrence
    (1, 8, 130, 32, 3, 0.03, [117], 1e-3),        # sharp plans, inside the factors' range
    (1, 8, 130, 32, 3, 0.003, [117], 1e-3),       # factors out of range: the general sweeps
    (1, 16, 256, 32, 20, 0.003, None, 1e-3),
])
def test_register_balanced_gradients(B, H, N, d, K, eps, lengths, tol):
    from deepfold_amd import balanced_sinkhorn_transport_dual

    print(f"case B{B} H{H} N{N} d{d} K{K} eps{eps}", flush=True)
    g = torch.Generator().manual_seed(N + K)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    leaves = dict(Q=unit(torch.randn(B, H, N, d, generator=g)), K=unit(torch.randn(B, H, N, d, generator=g)),
                  x=3 * torch.randn(B, N, 3, generator=g), V=torch.randn(B, H, N, d, generator=g),
                  al=-1 + 0.3 * torch.randn(H, generator=g), r=10 + torch.randn(H, generator=g))
    e, mask = torch.full((H,), eps), None
    if lengths is not None:
        mask = torch.zeros(B, N)
        for b, n in enumerate(lengths):
            mask[b, :n] = 1
    wx, wh = torch.randn(B, H, N, 3, generator=g), torch.randn(B, H, N, d, generator=g)
    if eps < 0.03:  # u of the last iteration against the initial zero: a row factor
        n = lengths[0] if lengths else N
        f = lambda t: t[:, :, :n].double()
        u = bt.sinkhorn_cpu(f(leaves["Q"]), f(leaves["K"]), leaves["x"][:, :n].double(), e.double(), leaves["al"].double(),
                            leaves["r"].double(), None, n, K, return_plan=True)[2]
        assert float(u.abs().amax(-1).min()) > MAX_FACTOR  # every head
    grads = []
    for fn, conv in ((bt.balanced_transport_dual, lambda t: None if t is None else t.double()),
                     (balanced_sinkhorn_transport_dual, lambda t: None if t is None else t.to(DEV))):
        p = {k: conv(v).requires_grad_(True) for k, v in leaves.items()}
        xc, hc = fn(p["Q"], p["K"], p["x"], p["V"], conv(e), p["al"], p["r"], K_iter=K, mask=conv(mask))
        ((xc * conv(wx)).sum() + (hc * conv(wh)).sum()).backward()
        grads.append({k: v.grad.detach().cpu().double().numpy() for k, v in p.items()})
    for k in leaves:
        assert_close_rel(grads[1][k], grads[0][k], tol, "d" + k)


@pytest.mark.parametrize("B,H,N,d,K,lengths", [
    (1, 4, 17, 32, 1, None),            # one iteration
    (2, 8, 150, 32, 33, [150, 90]),     # odd count, several batches of factors; warm start
    (1, 2, 40, 24, 65, None),           # past the kept iterations: the general sweeps
])
def test_register_unrolled_gradients(B, H, N, d, K, lengths):
    from deepfold_amd import flash_sinkhorn_attn
    from oracle import sinkhorn_dense_ref as dref

    print(f"case B{B} H{H} N{N} d{d} K{K}", flush=True)
    t = _uot(B, H, N, d, K, N + K, 0.3, lengths or [N] * B)
    names = ("Q", "K", "V", "G", "log_mu", "log_nu")
    go = torch.randn(B, N, H * d, generator=torch.Generator().manual_seed(3)) * t["mask"][:, :, None]
    want = {k: np.zeros(t[k].shape) for k in names}
    for b, n in enumerate(lengths or [N] * B):
        p = {k: t[k][b:b + 1, :, :n].double().clone().requires_grad_(True) for k in names}
        C = -(p["Q"] @ p["K"].transpose(-1, -2)) / math.sqrt(d)
        lu, lv = dref.sinkhorn_solve(C, p["log_mu"], p["log_nu"], t["eps"].double(), K=K,
                                     log_v_init=t["log_v_init"][b:b + 1, :, :n].double())
        o, _, _ = dref.compute_transport_output(p["V"], p["G"], lu, lv, C, t["eps"].double())
        (o * go[b:b + 1, :n].double()).sum().backward()
        for k in names:
            want[k][b:b + 1, :, :n] = p[k].grad.numpy()
    c = {k: v.to(DEV) for k, v in t.items()}
    p = {k: c[k].detach().requires_grad_(True) for k in names}
    o = flash_sinkhorn_attn(p["Q"], p["K"], p["V"], p["G"], c["x_res"], c["pos_weight"], None, c["eps"], None,
                            p["log_mu"], p["log_nu"], K_iter=K, log_v_init=c["log_v_init"], mask=c["mask"],
                            ift_mode="unrolled")[0]
    o.backward(go.to(DEV))
    for k in names:
        assert_close_rel(p[k].grad.cpu().double().numpy(), want[k], 1e-4, "d" + k)


@pytest.mark.parametrize("solver,iters,mode", [
    ("fixed_point", 4, "reference"), ("fixed_point", 0, "reference"), ("cg", 20, "reference"), ("cg", 20, "analytic"),
])
@pytest.mark.parametrize("B,H,N,d,v_scale,geo,lengths,dtype,tol", [
    (1, 2, 17, 32, 0.0, True, None, torch.float32, 1e-4),          # members without a tile
    (2, 8, 300, 24, 0.0, False, [300, 161], torch.float32, 1e-4),  # three tiles a member; padded columns
    (1, 4, 150, 32, 0.0, True, None, torch.bfloat16, 2e-2),
    (1, 4, 90, 32, 60.0, True, None, torch.float32, 1e-3),         # row sums out of range: the general sweeps
])
def test_register_ift_gradients(B, H, N, d, v_scale, geo, lengths, dtype, tol, solver, iters, mode):
    from test_gpu_sinkhorn_bwd import compare, grad_inputs, run_gpu_bwd
    from test_gpu_sinkhorn_fwd import make_inputs, oracle_inputs

    print(f"case B{B} H{H} N{N} d{d} v{v_scale} geo={geo} {dtype} {solver} {iters} {mode}", flush=True)
    inp = make_inputs(B, H, N, d, seed=N + d, eps=[1.0, 0.7] * (H // 2), pos_geo=geo)
    go, gxc = grad_inputs(B, H, N, d, seed=N + 1, with_xc=lengths is None)
    K, mask, kw = 6, None, {}
    if lengths is not None:
        mask = torch.zeros(B, N)
        for b, n in enumerate(lengths):
            mask[b, :n] = 1
        go = go * mask[:, :, None]
    oi = dict(oracle_inputs(inp, dtype))
    if v_scale:
        K = 1
        v0 = v_scale * torch.randn(B, H, N, generator=torch.Generator().manual_seed(4))
        kw["log_v_init"] = v0.to(DEV)
        oi["log_v_init"] = v0.numpy()
    got = run_gpu_bwd(inp, K, dtype, go, gxc, mask=mask, ift_solver=solver, ift_iters=iters, ift_mode=mode, **kw)
    gx = None if gxc is None else gxc.numpy()
    oi["K_iter"] = K
    if mask is not None:
        _, want = ref.backward_masked(dict(oi, mask=mask.numpy(), lam=1.0, r_0=10.0), go.numpy(), gx, mode=mode,
                                      solver=solver, n_cg=iters, K_back=iters)
    else:
        fo = ref.forward(**oi)
        if mode == "analytic":
            want = ref.backward_analytic(oi, fo, go.numpy(), gx)
        else:
            want = ref.backward_reference(oi, fo, go.numpy(), gx, K_back=iters, solver=solver, n_cg=iters)
    compare(got, want, tol, f"ift-{mode}-{solver}", skip=() if mask is None else ("pos_weight", "w_dist", "x_res"))


@pytest.mark.parametrize("solver,iters,mode", [
    ("fixed_point", 4, "reference"), ("fixed_point", 0, "reference"), ("fixed_point", 20, "analytic"),
    ("cg", 10, "reference"),
])
@pytest.mark.parametrize("geo,dtype,tol", [(False, torch.float32, 1e-4), (True, torch.float32, 1e-4),
                                           (True, torch.bfloat16, 2e-2)])
def test_register_ift_large_row_sums(geo, dtype, tol, solver, iters, mode):
    """Row sums near the top of the register form's range (log Z of 20 nats, the range ends at 22.2) and a
    last tile that the sequence does not fill: the entries past its end take part in no sum."""
    from test_gpu_sinkhorn_bwd import compare, grad_inputs, run_gpu_bwd
    from test_gpu_sinkhorn_fwd import make_inputs, oracle_inputs

    B, H, N, d, K = 1, 2, 90, 32, 1
    print(f"case geo={geo} {dtype} {solver} {iters} {mode}", flush=True)
    inp = make_inputs(B, H, N, d, seed=91, eps=[1.0, 1.0], pos_geo=geo)
    v0 = torch.full((B, H, N), -90.0)
    go, gxc = grad_inputs(B, H, N, d, seed=92, with_xc=True)
    oi = dict(oracle_inputs(inp, dtype), log_v_init=v0.numpy(), K_iter=K)
    fo = ref.forward(**oi)
    logz = []
    for h in range(H):
        z = ref._plan_pieces(oi["Q"][0, h], oi["K"][0, h], oi["x_res"][0], oi["pos_weight"][h],
                             None if oi["pos_bins"] is None else oi["pos_bins"][0], oi["w_dist"][h], 10.0,
                             oi["eps"][h], fo["log_u"][0, h], fo["log_v"][0, h])
        logz.append(z["logZ"])
        # v + column LSE = log nu - eps / lam v: both factors inside the range, so that no group leaves the form
        assert np.max(np.abs(oi["log_nu"][0, h] - fo["log_v"][0, h])) < MAX_FACTOR
    assert np.max(logz) < MAX_FACTOR and np.max(logz) > 19.7  # 2^128 / 1e30 in nats: the product that overflowed
    got = run_gpu_bwd(inp, K, dtype, go, gxc, ift_solver=solver, ift_iters=iters, ift_mode=mode,
                      log_v_init=v0.to(DEV))
    for k, v in got.items():
        assert np.isfinite(v).all(), k
    if mode == "analytic":
        want = ref.backward_analytic(oi, fo, go.numpy(), gxc.numpy())
    else:
        want = ref.backward_reference(oi, fo, go.numpy(), gxc.numpy(), K_back=iters, solver=solver, n_cg=iters)
    # (the analytic oracle solves the system exactly: 20 sweeps leave a share of kappa^40 = 2^-40)
    compare(got, want, tol, f"large-row-sums-{mode}-{solver}")


@pytest.mark.parametrize("op,geo", [("fixed_point", False), ("fixed_point", True), ("cg", False), ("cg", True),
                                    ("unrolled", False), ("unrolled", True), ("balanced", True)])
def test_gradients_ignore_padded_inputs(op, geo):
    """What padded rows hold, NaN included, changes no output and no gradient."""
    from deepfold_amd import balanced_sinkhorn_transport_dual, flash_sinkhorn_attn

    print(f"case {op} geo={geo}", flush=True)
    B, H, N, d, lengths = 2, 4, 90, 32, [83, 50]
    t = _uot(B, H, N, d, 5, 17, 0.0, lengths)
    g = torch.Generator().manual_seed(18)
    bins = torch.randint(0, 68, (B, N, N), generator=g, dtype=torch.int32).to(DEV) if geo else None
    t.update(pos_weight=0.3 * torch.randn(H, 68, generator=g), w_dist=torch.rand(H, generator=g),
             alpha=torch.full((H,), -1.0), r=torch.full((H,), 10.0))
    m = t["mask"].to(DEV)
    gx = torch.randn(B, H, N, 3, generator=g).to(DEV) * m[:, None, :, None]
    go = torch.randn(B, N, H * d, generator=g).to(DEV) * m[:, :, None]
    runs = []
    for fill in (0.0, float("nan")):
        c = {k: v.to(DEV).clone() for k, v in t.items()}
        for k in ("Q", "K", "V", "G"):
            c[k] = torch.where(m[:, None, :, None] > 0, c[k], torch.full_like(c[k], fill))
        c["x_res"] = torch.where(m[:, :, None] > 0, c["x_res"], torch.full_like(c["x_res"], fill))
        if op == "balanced":
            names = ("Q", "K", "x_res", "V", "alpha", "r")
            p = {k: c[k].requires_grad_(True) for k in names}
            out = balanced_sinkhorn_transport_dual(p["Q"], p["K"], p["x_res"], p["V"], c["eps"], p["alpha"], p["r"],
                                                   K_iter=5, mask=m)
            seeds = [gx, go.view(B, N, H, d).permute(0, 2, 1, 3).contiguous()]
        else:
            names = ("Q", "K", "V", "G", "x_res", "log_mu", "log_nu") + (("w_dist",) if geo else ())
            p = {k: c[k].requires_grad_(True) for k in names}
            kw = {"ift_mode": "unrolled"} if op == "unrolled" else {"ift_solver": op, "ift_iters": 6}
            out = flash_sinkhorn_attn(p["Q"], p["K"], p["V"], p["G"], p["x_res"], c["pos_weight"], bins, c["eps"],
                                      p.get("w_dist"), p["log_mu"], p["log_nu"], K_iter=5, mask=m, **kw)[:2]
            seeds = [go, gx]
        grads = torch.autograd.grad(list(out), list(p.values()), seeds)
        runs.append(dict(zip(names, grads), **{f"out{i}": o.detach() for i, o in enumerate(out)}))
    for k, want in runs[0].items():
        assert torch.isfinite(want).all(), k
        assert torch.equal(runs[1][k], want), k
