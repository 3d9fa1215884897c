"""GPU parity of the flash-Sinkhorn IFT backward against the CPU oracle and the
reference's own golden gradients.

Relative error = max |gpu - oracle| / max |oracle| per tensor; bars 1e-4 (fp32)
and 2e-2 (bf16) as in the north star.  Gradients that are pure cancellation
noise in the reference (d pos_weight / d w_dist when the position and geometry
terms are identically zero) are compared against an absolute floor instead.
"""

import glob
import os

import numpy as np
import pytest
import torch

from conftest import assert_close_rel, max_rel_err
from oracle import sinkhorn as ref
from test_gpu_sinkhorn_fwd import geometry_rounded, make_inputs, oracle_inputs

pytestmark = pytest.mark.gpu

GRADS = ("Q", "K", "V", "G", "x_res", "pos_weight", "w_dist", "log_mu", "log_nu")


def run_gpu_bwd(inp, K_iter, dtype, grad_o, grad_xc=None, mask=None, **kw):
    from deepfold_amd import flash_sinkhorn_attn

    dev = torch.device("cuda:0")
    leaves = {}
    t = {}
    for k, v in inp.items():
        if v is None:
            t[k] = None
            continue
        v = v.to(dev)
        if k in ("Q", "K", "V", "G"):
            v = v.to(dtype)
        if k in GRADS:
            v = v.clone().requires_grad_(True)
            leaves[k] = v
        t[k] = v
    o, xc, lu, lv = flash_sinkhorn_attn(t["Q"], t["K"], t["V"], t["G"], t["x_res"], t["pos_weight"], t["pos_bins"],
                                        t["eps"], t["w_dist"], t["log_mu"], t["log_nu"], K_iter=K_iter,
                                        mask=None if mask is None else mask.to(dev), **kw)
    loss = (o * grad_o.to(dev)).sum()
    if grad_xc is not None:
        loss = loss + (xc * grad_xc.to(dev)).sum()
    loss.backward()
    torch.cuda.synchronize()
    return {k: v.grad.float().cpu().numpy() for k, v in leaves.items()}


def compare(got, want, tol, label, skip=()):
    scale = max(float(np.max(np.abs(want[k]))) for k in ("Q", "K", "V"))
    for k in GRADS:
        if k in skip or k not in got:
            continue
        w = np.asarray(want[k])
        if float(np.max(np.abs(w))) < 1e-4 * scale:
            # cancellation-noise gradient: compare on the scale of the large ones
            err = float(np.max(np.abs(got[k] - w))) / scale
            assert err <= tol, f"{label}:{k} abs err {err:.3e} (relative to grad scale)"
        else:
            assert_close_rel(got[k], w, tol, f"{label}:{k}")


def grad_inputs(B, H, N, d, seed, with_xc=False):
    g = torch.Generator().manual_seed(seed)
    go = torch.randn(B, N, H * d, generator=g)
    gxc = torch.randn(B, H, N, 3, generator=g) if with_xc else None
    return go, gxc


@pytest.mark.parametrize("B,H,N,d,eps,K", [
    (1, 2, 48, 32, [0.5, 1.0], 6),
    (2, 2, 70, 16, [0.5, 2.0], 7),
    (1, 4, 256, 32, [1.0] * 4, 20),
    (1, 2, 100, 64, [0.25, 1.0], 5),
])
def test_backward_reference_fp32(B, H, N, d, eps, K):
    inp = make_inputs(B, H, N, d, seed=200 + N, eps=eps)
    go, gxc = grad_inputs(B, H, N, d, seed=300 + N, with_xc=True)
    got = run_gpu_bwd(inp, K, torch.float32, go, gxc)
    oi = oracle_inputs(inp, torch.float32)
    fo = ref.forward(**oi, K_iter=K)
    want = ref.backward_reference(dict(oi, K_iter=K), fo, go.numpy(), gxc.numpy())
    compare(got, want, 1e-4, "fp32-ref")


def test_backward_golden_vectors():
    """Gradients written by the reference's FlashSinkhornAttn.backward (tests/golden)."""
    here = os.path.dirname(os.path.abspath(__file__))
    files = sorted(glob.glob(os.path.join(here, "golden", "flash_sinkhorn_*.npz")))
    assert files
    for f in files:
        z = np.load(f)
        inp = {k: torch.from_numpy(z[k]) for k in ("Q", "K", "V", "G", "x_res", "pos_weight", "pos_bins",
                                                   "eps", "w_dist", "log_mu", "log_nu")}
        got = run_gpu_bwd(inp, int(z["K_iter"]), torch.float32, torch.from_numpy(z["grad_o"]),
                          torch.from_numpy(z["grad_xc"]))
        want = {k: z["grad_" + k] for k in GRADS}
        # torch.cdist's matmul path (N > 25) rounds the reference's forward distances:
        # with geometry on (ragged_tile, N = 70) the CPU oracle itself differs from these
        # vectors by 5e-4 in d w_dist, so that file gets 1e-3; the others the fp32 bar 1e-4.
        tol = 1e-3 if geometry_rounded(z) else 1e-4
        compare(got, want, tol, os.path.basename(f))


def test_cg_matches_converged_fixed_point():
    """CG and the reference fixed point solve the same system (agree <= 1e-5 on z)."""
    B, H, N, d = 1, 2, 96, 32
    inp = make_inputs(B, H, N, d, seed=41, eps=[0.5, 0.5])
    go, _ = grad_inputs(B, H, N, d, seed=42)
    fp = run_gpu_bwd(inp, 30, torch.float32, go, ift_solver="fixed_point", ift_iters=60)
    cg = run_gpu_bwd(inp, 30, torch.float32, go, ift_solver="cg", ift_iters=30)
    # kappa = 2/3: 60 Gauss-Seidel sweeps contract by (4/9)^60; CG converges in << 30 steps.
    # z_v (d log_nu) agrees to 1e-5; z_u = kappa S_col z_v is a cancelling sum whose fp32
    # rounding differs between the two solvers (~2e-5), so it and the gradients get 1e-4.
    assert max_rel_err(cg["log_nu"], fp["log_nu"]) <= 1e-5
    assert max_rel_err(cg["log_mu"], fp["log_mu"]) <= 1e-4
    for k in ("Q", "K", "V"):
        assert max_rel_err(cg[k], fp[k]) <= 1e-4, k


def test_cg_matches_oracle_cg():
    B, H, N, d = 1, 2, 64, 32
    inp = make_inputs(B, H, N, d, seed=51, eps=[0.5, 0.25])
    go, gxc = grad_inputs(B, H, N, d, seed=52, with_xc=True)
    got = run_gpu_bwd(inp, 20, torch.float32, go, gxc, ift_solver="cg", ift_iters=20)
    oi = oracle_inputs(inp, torch.float32)
    fo = ref.forward(**oi, K_iter=20)
    want = ref.backward_reference(dict(oi, K_iter=20), fo, go.numpy(), gxc.numpy(), solver="cg", n_cg=20)
    compare(got, want, 1e-4, "cg")


def test_analytic_mode_matches_oracle():
    B, H, N, d = 1, 2, 48, 32
    inp = make_inputs(B, H, N, d, seed=61, eps=[0.5, 1.0])
    go, gxc = grad_inputs(B, H, N, d, seed=62, with_xc=True)
    got = run_gpu_bwd(inp, 40, torch.float32, go, gxc, ift_solver="cg", ift_iters=40, ift_mode="analytic")
    oi = oracle_inputs(inp, torch.float32)
    fo = ref.forward(**oi, K_iter=40)
    want = ref.backward_analytic(dict(oi, K_iter=40), fo, go.numpy(), gxc.numpy())
    compare(got, want, 1e-4, "analytic")


@pytest.mark.parametrize("solver,iters", [("fixed_point", None), ("cg", 20)])
def test_backward_masked_bf16(solver, iters):
    """Ragged batch with padding mask == per-sample unpadded evaluation (bf16 bar)."""
    B, H, N, d = 2, 2, 96, 32
    K = 12
    inp = make_inputs(B, H, N, d, seed=71, eps=[0.5, 1.0])
    go, _ = grad_inputs(B, H, N, d, seed=72)
    lengths = [96, 61]
    mask = torch.zeros(B, N)
    for b, n in enumerate(lengths):
        mask[b, :n] = 1
        go[b, n:] = 0
    got = run_gpu_bwd(inp, K, torch.bfloat16, go, None, mask=mask, ift_solver=solver, ift_iters=iters)
    oi = oracle_inputs(inp, torch.bfloat16)
    oi["mask"] = mask.numpy()
    _, want = ref.backward_masked(dict(oi, K_iter=K, lam=1.0, r_0=10.0), go.numpy(), None,
                                  solver=solver, n_cg=iters)
    compare(got, want, 2e-2, f"masked-{solver}", skip=("pos_weight", "w_dist", "x_res"))
    for b, n in enumerate(lengths):
        for k in ("Q", "K", "V", "G"):
            assert np.all(got[k][b, :, n:] == 0), k


def test_backward_general_cost_fp32():
    """Position bins + geometry: d pos_weight, d w_dist and d x_res through the cost."""
    B, H, N, d = 2, 2, 40, 32
    inp = make_inputs(B, H, N, d, seed=81, eps=[0.5, 2.0], pos_geo=True)
    go, gxc = grad_inputs(B, H, N, d, seed=82, with_xc=True)
    got = run_gpu_bwd(inp, 5, torch.float32, go, gxc)
    oi = oracle_inputs(inp, torch.float32)
    fo = ref.forward(**oi, K_iter=5)
    want = ref.backward_reference(dict(oi, K_iter=5), fo, go.numpy(), gxc.numpy())
    compare(got, want, 1e-4, "general")


def test_backward_bins_outside_table():
    """Bins outside [0, 68) carry no bias and receive no d pos_weight: the gradients
    equal the oracle's with a 69-entry table (entry 68 = 0) and those bins remapped
    to 68, whose extra gradient entry is dropped."""
    B, H, N, d = 2, 2, 40, 32
    inp = make_inputs(B, H, N, d, seed=83, eps=[0.5, 2.0], pos_geo=True)
    g = torch.Generator().manual_seed(84)
    bins = inp["pos_bins"].clone()
    sel = torch.rand(bins.shape, generator=g) < 0.2
    bad = torch.tensor([-1, 68, 200, 1 << 20], dtype=torch.int32)[torch.randint(0, 4, bins.shape, generator=g)]
    bins[sel] = bad[sel]
    inp["pos_bins"] = bins
    go, gxc = grad_inputs(B, H, N, d, seed=85, with_xc=True)
    got = run_gpu_bwd(inp, 5, torch.float32, go, gxc)
    oi = oracle_inputs(inp, torch.float32)
    oi["pos_weight"] = np.concatenate([oi["pos_weight"], np.zeros((H, 1), np.float32)], 1)
    b = oi["pos_bins"].astype(np.int64)
    b[(b < 0) | (b >= 68)] = 68
    oi["pos_bins"] = b
    fo = ref.forward(**oi, K_iter=5)
    want = ref.backward_reference(dict(oi, K_iter=5), fo, go.numpy(), gxc.numpy())
    compare(got, want, 1e-4, "bins-outside", skip=("pos_weight",))
    assert_close_rel(got["pos_weight"], np.asarray(want["pos_weight"])[:, :68], 1e-4, "bins-outside:pos_weight")


# (d = 32 keeps the plan in registers and reads no matrix; d = 64 does)
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("dtype,solver", [(torch.float32, "cg"), (torch.bfloat16, "fixed_point")])
def test_backward_precomputed_bias_matches_per_element(dtype, solver, d):
    """With the workspace extension (dfl_sinkhorn_bias_workspace_size) the backward
    evaluates the position / geometry bias once and reads it in its sweeps; without it
    every sweep evaluates bins and distances.  Both read the same values, so the
    gradients of Q, K, V, G and the marginals are bit-identical (ragged lengths, masked
    tokens, bins outside the table); d pos_weight, d w_dist and d x_res reduce through
    LDS atomics whose order varies from run to run, so they agree to fp32 rounding."""
    import importlib

    from deepfold_amd import _lib

    fsa = importlib.import_module("deepfold_amd.flash_sinkhorn_attn")  # the module, not the function

    B, H, N = 2, 3, 200
    inp = make_inputs(B, H, N, d, seed=91, eps=[0.5, 1.0, 2.0], pos_geo=True)
    g = torch.Generator().manual_seed(92)
    bins = inp["pos_bins"].clone()
    bins[torch.rand(bins.shape, generator=g) < 0.1] = 77
    inp["pos_bins"] = bins
    mask = torch.ones(B, N)
    mask[0, 150:] = 0
    mask[1, 17] = 0
    go, gxc = grad_inputs(B, H, N, d, seed=93, with_xc=True)
    go = go * mask[:, :, None]
    kw = dict(ift_solver=solver, ift_iters=12 if solver == "cg" else None)
    got, sizes = {}, {}
    saved = fsa._BIAS_WS_MAX
    try:
        for label, cap in (("matrix", saved), ("per_element", -1)):
            fsa._BIAS_WS_MAX = cap
            _lib._ws_cache.clear()  # the next workspace is exactly the requested size
            got[label] = run_gpu_bwd(inp, 6, dtype, go, gxc, mask=mask, **kw)
            sizes[label] = max(w.numel() for w in _lib._ws_cache.values())
    finally:
        fsa._BIAS_WS_MAX = saved
        _lib._ws_cache.clear()
    assert (sizes["matrix"] > sizes["per_element"]) == (d == 64)
    for k in got["matrix"]:
        if k in ("pos_weight", "w_dist", "x_res"):
            assert max_rel_err(got["matrix"][k], got["per_element"][k]) <= 1e-6, k
        else:
            assert np.array_equal(got["matrix"][k], got["per_element"][k]), k
    assert all(np.isfinite(v).all() for v in got["matrix"].values())
