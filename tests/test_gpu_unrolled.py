"""GPU parity of the unrolled flash-Sinkhorn backward (``ift_mode="unrolled"``,
the default of ``flash_sinkhorn``) against autograd through the dense float64
iteration: oracle/sinkhorn_dense_ref.py (sinkhorn_solve + compute_transport_output)
on the flash cost built here, which is what the reference's
tests/test_triton_fallback_consistency.py:312-430 checks its Triton unrolled
backward against (at 5e-3; the bar here is 1e-4 in fp32, 2e-2 in bf16).

Cases: the reference test's shapes (B1 H2 N16 d32 K3; B2 masked), a gated
ragged batch with position bins, geometry and a warm start, bf16 inputs at
d = 64, and a longer sequence whose members own several tiles.
"""

import numpy as np
import pytest
import torch

from conftest import assert_close_rel
from oracle import sinkhorn_dense_ref as dref

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _inputs(B, H, N, d, seed, eps, lens=None, warm=False):
    g = torch.Generator().manual_seed(seed)
    t = dict(Q=torch.randn(B, H, N, d, generator=g) / d ** 0.5 * 2, K=torch.randn(B, H, N, d, generator=g) / d ** 0.5,
             V=torch.randn(B, H, N, d, generator=g), G=torch.randn(B, H, N, d, generator=g),
             x=torch.randn(B, N, 3, generator=g) * 3, pw=torch.randn(H, 68, generator=g) * 0.3,
             wd=torch.rand(H, generator=g),
             lmu=torch.log_softmax(torch.randn(B, H, N, generator=g), -1),
             lnu=torch.log_softmax(torch.randn(B, H, N, generator=g), -1))
    bins = torch.randint(0, 68, (B, N, N), generator=g, dtype=torch.int32)
    if warm:
        t["v0"] = 0.3 * torch.randn(B, H, N, generator=g)
    mask = None
    if lens is not None:
        mask = torch.zeros(B, N)
        for b, n in enumerate(lens):
            mask[b, :n] = 1
    wo = torch.randn(B, N, H * d, generator=g)
    wx = torch.randn(B, H, N, 3, generator=g)
    return t, bins, torch.tensor(eps, dtype=torch.float32), mask, wo, wx


def _oracle(t, bins, eps, mask, wo, wx, K, r0=10.0, lam=1.0):
    L = {k: v.double().clone().requires_grad_(True) for k, v in t.items()}
    B, H, N, d = L["Q"].shape
    dist = (L["x"][:, :, None] - L["x"][:, None, :]).norm(dim=-1).clamp(min=1e-8)
    C = (-(L["Q"] @ L["K"].transpose(-1, -2)) / d ** 0.5 + L["pw"][:, bins.long()].permute(1, 0, 2, 3)
         + L["wd"][None, :, None, None] * (dist / (r0 + dist))[:, None])
    m = None if mask is None else mask.double()
    lu, lv = dref.sinkhorn_solve(C, L["lmu"], L["lnu"], eps.double(), lam=lam, K=K, log_v_init=L.get("v0"), mask=m)
    o, _, xc = dref.compute_transport_output(L["V"], L["G"], lu, lv, C, eps.double(), L["x"], m)
    ((o * wo.double()).sum() + (xc * wx.double()).sum()).backward()
    return {"o": o, "xc": xc, "lu": lu, "lv": lv}, {k: v.grad for k, v in L.items()}


def _gpu(t, bins, eps, mask, wo, wx, K, dtype, r0=10.0, lam=1.0):
    from deepfold_amd import flash_sinkhorn_attn

    L = {k: v.to(DEV) for k, v in t.items()}
    for k in ("Q", "K", "V", "G"):
        L[k] = L[k].to(dtype)
    L = {k: v.detach().requires_grad_(True) for k, v in L.items()}
    o, xc, lu, lv = flash_sinkhorn_attn(L["Q"], L["K"], L["V"], L["G"], L["x"], L["pw"], bins.to(DEV), eps.to(DEV),
                                        L["wd"], L["lmu"], L["lnu"], K_iter=K, lam=lam, r_0=r0,
                                        log_v_init=L.get("v0"), mask=None if mask is None else mask.to(DEV),
                                        ift_mode="unrolled")
    ((o * wo.to(DEV)).sum() + (xc * wx.to(DEV)).sum()).backward()
    return {"o": o, "xc": xc, "lu": lu, "lv": lv}, {k: v.grad for k, v in L.items()}


CASES = [
    # B, H, N, d, K, eps, lens, warm, dtype, tol
    (1, 2, 16, 32, 3, [0.5, 1.0], None, False, torch.float32, 1e-4),          # reference test_backward_unbatched
    (2, 2, 16, 32, 3, [0.5, 1.0], [16, 11], False, torch.float32, 1e-4),      # reference batched masked
    (2, 3, 70, 32, 7, [0.5, 1.0, 2.0], [70, 41], False, torch.float32, 1e-4),  # gate, bins, geometry, ragged
    # warm start at K = 3: d log_v_init decays geometrically with K (about 1e-12 at K = 7,
    # below fp32 rounding of the other gradients), so it is compared where it is measurable
    (2, 3, 70, 32, 3, [0.5, 1.0, 2.0], [70, 41], True, torch.float32, 1e-4),
    (1, 2, 48, 64, 5, [0.7, 1.3], None, False, torch.bfloat16, 2e-2),
    (1, 2, 300, 32, 4, [0.5, 1.0], [290], False, torch.float32, 1e-4),        # several tiles per member
    # bf16 with d <= 32
    (2, 3, 70, 32, 5, [0.5, 1.0, 2.0], [70, 41], False, torch.bfloat16, 2e-2),
    (1, 2, 300, 32, 4, [0.5, 1.0], [290], False, torch.bfloat16, 2e-2),
]


@pytest.mark.parametrize("B,H,N,d,K,eps,lens,warm,dtype,tol", CASES)
def test_unrolled_matches_dense_autograd(B, H, N, d, K, eps, lens, warm, dtype, tol):
    print(f"case B{B} H{H} N{N} d{d} K{K} {dtype}", flush=True)
    t, bins, e, mask, wo, wx = _inputs(B, H, N, d, seed=N * 7 + K, eps=eps, lens=lens, warm=warm)
    if dtype == torch.bfloat16:  # the oracle sees the rounded values
        for k in ("Q", "K", "V", "G"):
            t[k] = t[k].to(torch.bfloat16).float()
    vr, gr = _oracle(t, bins, e, mask, wo, wx, K)
    vg, gg = _gpu(t, bins, e, mask, wo, wx, K, dtype)
    for k in ("o", "xc", "lu", "lv"):
        assert_close_rel(vg[k].detach().float().cpu().numpy(), vr[k].detach().numpy(), tol, k)
    for k, want in gr.items():
        got = gg[k]
        assert got is not None, k
        got = got.float().cpu().numpy()
        assert np.isfinite(got).all(), k
        if k == "v0":
            # d log_v_init = -kappa (s^{R,0})^T gl_u^0 sums terms of both signs that nearly
            # cancel (it is ~1e-2 of the other potential gradients at K = 3): its fp32
            # error is held to the bar relative to the scale of d log_nu, a gradient of
            # the same kind, rather than to its own small maximum
            scale = max(float(np.abs(want.numpy()).max()), float(np.abs(gr["lnu"].numpy()).max()))
            err = float(np.abs(got - want.numpy()).max()) / scale
            assert err <= tol, f"grad v0: error {err:.3e} of the d log_nu scale > {tol:.1e}"
            continue
        assert_close_rel(got, want.numpy(), tol, f"grad {k}")


def test_flash_sinkhorn_defaults_to_unrolled():
    """flash_sinkhorn (sinkhorn_kernel.py:2385) differentiates through the iterations
    by default, as the reference's; FlashSinkhornFunction.apply likewise."""
    from deepfold_amd import FlashSinkhornFunction, flash_sinkhorn

    B, H, N, d, K = 1, 2, 24, 32, 4
    t, bins, e, _, _, wx = _inputs(B, H, N, d, seed=5, eps=[0.5, 1.0])
    g = torch.Generator().manual_seed(6)
    wO = torch.randn(B, H, N, d, generator=g)
    t["G"] = torch.full_like(t["G"], 30.0)  # sigma = 1 - 9e-14: the gated oracle is the ungated op
    vr, gr = _oracle(t, bins, e, None, wO.permute(0, 2, 1, 3).reshape(B, N, H * d), wx, K)
    for fn in ("flash_sinkhorn", "apply"):
        L = {k: v.to(DEV).detach().requires_grad_(True) for k, v in t.items() if k != "G"}
        args = (L["Q"], L["K"], L["V"], L["x"], L["pw"], bins.to(DEV), e.to(DEV), L["wd"], L["lmu"], L["lnu"])
        if fn == "flash_sinkhorn":
            O, xc, _, _ = flash_sinkhorn(*args, K_iter=K)
        else:
            O, xc, _, _ = FlashSinkhornFunction.apply(*args, K, 1.0, 10.0, None, None, 64, None)
        ((O * wO.to(DEV)).sum() + (xc * wx.to(DEV)).sum()).backward()
        for k in ("Q", "K", "V", "x", "pw", "wd", "lmu", "lnu"):
            assert_close_rel(L[k].grad.cpu().numpy(), gr[k].numpy(), 1e-4, f"{fn} grad {k}")


def _content_only(B, H, N, d, K, lens, dtype, extreme=False):
    """Oracle and GPU results of the content-only cost (no bins, no geometry: the
    kernel's GEN = false build).  extreme: a few log-marginals at -70, which puts the
    ratio of a sweep's two exponentials outside the kernel's factored range (2^+-40),
    so those sweeps take the exact two-exponential path."""
    t, bins, e, mask, wo, wx = _inputs(B, H, N, d, seed=N + 3 * K, eps=[0.5] * H, lens=lens)
    t["pw"] = torch.zeros_like(t["pw"])
    t["wd"] = torch.zeros_like(t["wd"])
    if extreme:
        t["lmu"][..., :3] = -70.0
        t["lnu"][..., 5:8] = -70.0
    if dtype == torch.bfloat16:
        for k in ("Q", "K", "V", "G"):
            t[k] = t[k].to(torch.bfloat16).float()
    vr, gr = _oracle(t, torch.zeros_like(bins), e, mask, wo, wx, K)
    from deepfold_amd import flash_sinkhorn_attn

    L = {k: v.to(DEV) for k, v in t.items()}
    for k in ("Q", "K", "V", "G"):
        L[k] = L[k].to(dtype)
    L = {k: v.detach().requires_grad_(True) for k, v in L.items()}
    # no bins and w_dist = None (the reference's w_dist = 0 without reading x): GEN = false
    o, xc, lu, lv = flash_sinkhorn_attn(L["Q"], L["K"], L["V"], L["G"], L["x"], L["pw"], None, e.to(DEV), None,
                                        L["lmu"], L["lnu"], K_iter=K, mask=mask.to(DEV), ift_mode="unrolled")
    ((o * wo.to(DEV)).sum() + (xc * wx.to(DEV)).sum()).backward()
    return {"o": o, "xc": xc, "lu": lu, "lv": lv}, L, vr, gr


def _check(vg, L, vr, gr, tol):
    for k in ("o", "xc", "lu", "lv"):
        assert_close_rel(vg[k].detach().float().cpu().numpy(), vr[k].detach().numpy(), tol, k)
    for k in ("Q", "K", "V", "G", "lmu", "lnu"):
        got = L[k].grad.float().cpu().numpy()
        assert np.isfinite(got).all(), k
        assert_close_rel(got, gr[k].numpy(), tol, f"grad {k}")


# (2, 8, 768, ...) is the headline layout (B2 H8 N768, n_b = [501, 759]: two and three
# resident tiles per member, the plan in registers); N = 832 is past the register form, and
# resident operands would need 166752 bytes of LDS (over 160 KiB) there: Q and K from L2
@pytest.mark.parametrize("B,H,N,d,K,lens", [(2, 4, 96, 32, 6, [96, 61]), (1, 2, 300, 24, 4, [290]),
                                             (2, 8, 768, 32, 3, [501, 759]), (1, 2, 832, 32, 3, [829])])
def test_unrolled_content_only_bf16(B, H, N, d, K, lens):
    """The content-only cost (the build the headline workload runs) with bf16 inputs
    at d <= 32."""
    print(f"case content-only B{B} H{H} N{N} d{d} K{K}", flush=True)
    _check(*_content_only(B, H, N, d, K, lens, torch.bfloat16), 2e-2)


# B*H = 64 -> 4 members per head: 5-6 resident tiles per member (strided wave mapping,
# two tiles a wave on some SIMDs) and 8-10 (whole tiles per wave), more than the register
# form holds: the general sweeps, bf16 with Q and K resident in LDS, fp32 with both from L2
@pytest.mark.parametrize("N,lens,dtype,tol", [
    (384, [384, 350, 300, 330], torch.bfloat16, 2e-2),
    (640, [640, 600, 560, 530], torch.bfloat16, 2e-2),
    (384, [384, 350, 300, 330], torch.float32, 1e-4),
])
def test_unrolled_many_tiles_per_member(N, lens, dtype, tol):
    print(f"case many tiles B4 H16 N{N} {dtype}", flush=True)
    _check(*_content_only(4, 16, N, 32, 3, lens, dtype), tol)


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-4), (torch.bfloat16, 2e-2)])
def test_unrolled_exact_factor_path(dtype, tol):
    """Sweeps whose exponential ratio leaves the factored range take the exact path (the groups
    are out of the register form's range too: its kernel runs the general sweeps)."""
    print(f"case extreme marginals {dtype}", flush=True)
    _check(*_content_only(2, 2, 96, 32, 4, [96, 61], dtype, extreme=True), tol)


# (1, 2, 96): groups that leave the register form inside its kernel; (4, 16, 384): six resident
# tiles a member, the general sweeps in a kernel of their own, bf16 with resident Q and K
@pytest.mark.parametrize("extreme", [False, True])
@pytest.mark.parametrize("B,H,N,lens,K,dtype,tol", [
    (1, 2, 96, [90], 4, torch.float32, 1e-4),
    (1, 2, 96, [90], 4, torch.bfloat16, 2e-2),
    (4, 16, 384, [384, 350, 300, 330], 3, torch.bfloat16, 2e-2),
])
def test_unrolled_general_sweeps_full_cost(B, H, N, lens, K, dtype, tol, extreme):
    """Bins and geometry in the general sweeps, with and without marginals that put the exponential
    ratio outside the factored range."""
    print(f"case full cost B{B} H{H} N{N} K{K} {dtype} extreme={extreme}", flush=True)
    t, bins, e, mask, wo, wx = _inputs(B, H, N, 32, seed=N + 5, eps=[0.5, 1.0] * (H // 2), lens=lens)
    if extreme:
        t["lmu"][..., :3] = -70.0
        t["lnu"][..., 5:8] = -70.0
    if dtype == torch.bfloat16:
        for k in ("Q", "K", "V", "G"):
            t[k] = t[k].to(torch.bfloat16).float()
    vr, gr = _oracle(t, bins, e, mask, wo, wx, K)
    vg, gg = _gpu(t, bins, e, mask, wo, wx, K, dtype)
    for k in ("o", "xc", "lu", "lv"):
        assert_close_rel(vg[k].detach().float().cpu().numpy(), vr[k].detach().numpy(), tol, k)
    for k, want in gr.items():
        got = gg[k].float().cpu().numpy()
        assert np.isfinite(got).all(), k
        assert_close_rel(got, want.numpy(), tol, f"grad {k}")
