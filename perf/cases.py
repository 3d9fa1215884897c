"""The calls that this framework is timed and checked on.

``listed()`` names them, ``draw`` makes more of the same ranges.  A case is one pass
through the package's public functions as a model calls them: the unbalanced
flash-Sinkhorn attention (its implicit and its unrolled gradient, with and without the
position and geometry terms), the balanced transport alone and inside the block step,
the dense Sinkhorn, the diffusion attention, the windowed atom attention and the two
atom/token cross attentions.  Training cases return their outputs and every gradient.
``exact`` restates each pass in float64 torch.
"""

import math
import os
import sys
from types import SimpleNamespace

import torch

# the repository's root is the working folder; its package lies one folder below
_PKG = os.path.join(os.getcwd(), "deepfold-linear_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
BINS = 68      # position bins of the cost and of the diffusion attention
R0 = 10.0      # distance scale of the geometry term
ATOMS = 24     # atoms of a token, on average


def listed():
    return [
        # inference of one small attention layer: a short chain, where latency counts
        dict(name="uot_small", kind="uot", B=1, H=4, N=256, d=32, dtype="f32", K=20, eps=1.0, iters=0, full=False,
             ragged=False, train=False),
        # training of the attention layer on a padded batch, implicit gradient by CG: the usual call
        dict(name="uot_train", kind="uot", B=2, H=8, N=768, d=32, dtype="bf16", K=50, eps=0.5, iters=20, full=False,
             ragged=True, train=True),
        # the same layer with position bins and geometry, all defaults (7 iterations, fixed point), odd length
        dict(name="uot_full", kind="uot", B=1, H=16, N=389, d=32, dtype="bf16", K=7, eps=0.5, iters=0, full=True,
             ragged=False, train=True),
        # the longest sequence: a 4096-token complex, one sample
        dict(name="uot_large", kind="uot", B=1, H=16, N=4096, d=64, dtype="bf16", K=100, eps=0.25, iters=30,
             full=False, ragged=False, train=True),
        # flash_sinkhorn with its default gradient, through the executed iterations
        dict(name="unrolled", kind="unrolled", B=2, H=8, N=768, d=32, dtype="bf16", K=50, eps=0.5, full=False,
             ragged=True),
        # the transport inside a trunk block, alone
        dict(name="balanced", kind="balanced", B=1, H=16, N=256, d=32, K=20, ragged=False),
        # steps 2-4 of a trunk block: projections, transport, output projection, coordinates
        dict(name="block", kind="block", B=2, H=16, N=384, C=512, K=20, ragged=True),
        # the solver and output on a cost matrix that the caller built
        dict(name="dense", kind="dense", B=2, H=8, N=512, d=32, K=7, ragged=True),
        # training of the diffusion transformer: several noised copies, dense pair bias, gate
        dict(name="diffusion", kind="diffusion", B=4, H=16, N=1024, d=24, dtype="bf16", bias="dense", gate=True,
             ragged=False, train=True),
        # sampling with the position-bin bias, ragged length
        dict(name="diffusion_bins", kind="diffusion", B=1, H=16, N=777, d=32, dtype="bf16", bias="bins", gate=False,
             ragged=True, train=False),
        # atom encoder / decoder: windows of 32 queries and 128 keys with a bias of their own
        dict(name="window", kind="window", B=1, H=4, M=8192, d=32, dtype="bf16", bias=True, ragged=False, train=True),
        # atoms read from tokens and tokens from their atoms
        dict(name="cross", kind="cross", B=1, H=4, M=8192, d=32, dtype="bf16", train=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any of the calls, sizes spread over the logarithm of their range."""
    kind = rng.choice(["uot", "uot", "unrolled", "balanced", "block", "dense", "diffusion", "diffusion", "window",
                       "cross"])
    c = dict(kind=kind)
    if kind == "uot":
        c.update(B=rng.choice([1, 2, 4]), H=rng.choice([4, 8, 16]), N=_log(rng, 48, 1536), d=rng.choice([32, 64]),
                 dtype=rng.choice(["bf16", "bf16", "f32"]), K=rng.choice([7, 20, 50]), eps=rng.choice([0.25, 0.5, 1.0]),
                 iters=rng.choice([0, 20]), full=rng.random() < 0.5, ragged=rng.random() < 0.5,
                 train=rng.random() < 0.7)
        if c["N"] > 768:
            c.update(B=1, K=min(c["K"], 20))
    elif kind == "unrolled":
        c.update(B=rng.choice([1, 2]), H=rng.choice([4, 8, 16]), N=_log(rng, 48, 900), d=rng.choice([32, 64]),
                 dtype=rng.choice(["bf16", "f32"]), K=rng.choice([7, 20, 50]), eps=rng.choice([0.5, 1.0]),
                 full=rng.random() < 0.5, ragged=rng.random() < 0.5)
    elif kind == "balanced":
        c.update(B=rng.choice([1, 2, 4]), H=rng.choice([8, 16]), N=_log(rng, 48, 512), d=rng.choice([16, 32]),
                 K=rng.choice([10, 20]), ragged=rng.random() < 0.5)
    elif kind == "block":
        C, H = rng.choice([(512, 16), (256, 8), (128, 4)])
        c.update(B=rng.choice([1, 2, 4]), H=H, N=_log(rng, 48, 512), C=C, K=20, ragged=rng.random() < 0.5)
    elif kind == "dense":
        c.update(B=rng.choice([1, 2]), H=rng.choice([4, 8, 16]), N=_log(rng, 48, 900), d=rng.choice([16, 32, 64]),
                 K=rng.choice([7, 20]), ragged=rng.random() < 0.5)
    elif kind == "diffusion":
        c.update(B=rng.choice([1, 2, 4, 8]), H=rng.choice([4, 16]), N=_log(rng, 64, 1400), d=rng.choice([24, 32, 48]),
                 dtype=rng.choice(["bf16", "bf16", "f32"]), bias=rng.choice(["dense", "bins"]),
                 gate=rng.random() < 0.5, ragged=rng.random() < 0.5, train=rng.random() < 0.7)
        c["B"] = max(1, min(c["B"], (1 << 26) // (c["H"] * c["N"] * c["N"])))
    elif kind == "window":
        c.update(B=rng.choice([1, 2]), H=rng.choice([4, 8]), M=_log(rng, 256, 32768), d=32,
                 dtype=rng.choice(["bf16", "bf16", "f32"]), bias=rng.random() < 0.6, ragged=rng.random() < 0.5,
                 train=rng.random() < 0.7)
    else:
        c.update(B=rng.choice([1, 2]), H=rng.choice([4, 8]), M=_log(rng, 512, 16384), d=32,
                 dtype=rng.choice(["bf16", "bf16", "f32"]), train=rng.random() < 0.7)
    return c


def _lengths(case, n):
    """Valid tokens of each sample: a ragged batch keeps between about half and all of them."""
    B = case["B"]
    return [n - n // 85 - b * n // (2 * B) for b in range(B)] if case.get("ragged") else [n] * B


def _mask(case, n, dev):
    if not case.get("ragged"):
        return None
    m = torch.zeros(case["B"], n, device=dev)
    for b, k in enumerate(_lengths(case, n)):
        m[b, :k] = 1.0
    return m


def _chain(g, B, n, dev):
    """Residue coordinates: a random walk of 3.8 A steps, in the units of the distance scale."""
    step = torch.randn(B, n, 3, generator=g, device=dev)
    x = torch.cumsum(step / step.norm(dim=-1, keepdim=True).clamp(min=1e-3) * 3.8, dim=1)
    return (x - x.mean(dim=1, keepdim=True)).contiguous()


def _marginals(case, g, dev):
    """log mu, log nu: Dirichlet(5) weights on the valid tokens of training cases, uniform for inference."""
    B, H, N = case["B"], case["H"], case["N"]
    out = []
    for _ in range(2):
        t = torch.zeros(B, H, N, device=dev)
        for b, n in enumerate(_lengths(case, N)):
            if case.get("train", True):
                w = torch.zeros(H, n, device=dev)
                for _ in range(5):  # Gamma(5): a sum of five exponentials
                    w += -torch.log(torch.rand(H, n, generator=g, device=dev).clamp(min=1e-7))
                t[b, :, :n] = torch.log(w / w.sum(-1, keepdim=True))
            else:
                t[b, :, :n] = -math.log(n)
        out.append(t)
    return out


def prepare(case, seed):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(int(seed) * 7919 + 17)
    kind, B, H = case["kind"], case["B"], case["H"]
    dt = DTYPES[case.get("dtype", "f32")]

    def rnd(*shape, scale=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=g, device=dev) * scale).to(dtype)

    s = dict(case=case, p={}, const={}, grad=[])
    p, const = s["p"], s["const"]
    if kind in ("uot", "unrolled"):
        N, d = case["N"], case["d"]
        # layer-normalised queries and keys (unit variance a channel before the 1/sqrt(d) of the cost)
        p.update(Q=rnd(B, H, N, d, dtype=dt), K=rnd(B, H, N, d, dtype=dt), V=rnd(B, H, N, d, dtype=dt))
        if kind == "uot":
            p["G"] = rnd(B, H, N, d, dtype=dt)
        p["log_mu"], p["log_nu"] = _marginals(case, g, dev)
        const["eps"] = torch.full((H,), case["eps"], device=dev)
        const["mask"] = _mask(case, N, dev)
        x = _chain(g, B, N, dev)
        if case["full"]:
            i = torch.arange(N, device=dev)
            rel = (i[:, None] - i[None, :]).clamp(-32, 32) + 32
            other = torch.rand(B, N, N, generator=g, device=dev) < 0.05  # another chain: the last bins
            const["bins"] = torch.where(other, 65 + torch.randint(0, 3, (B, N, N), generator=g, device=dev),
                                        rel[None]).to(torch.int32).contiguous()
            p.update(x=x, pos_weight=rnd(H, BINS, scale=0.5), w_dist=torch.rand(H, generator=g, device=dev))
        else:
            const.update(bins=None, x=x, pos_weight=torch.zeros(H, BINS, device=dev))
        s["grad"] = [rnd(B, N, H * d) if kind == "uot" else rnd(B, H, N, d)]
        if case["full"]:
            s["grad"].append(rnd(B, H, N, 3, scale=0.3))
        if const["mask"] is not None:  # padded outputs reach no loss
            m = const["mask"]
            for k, t in enumerate(s["grad"]):
                s["grad"][k] = (t * (m[:, :, None] if t.dim() == 3 else m[:, None, :, None])).contiguous()
    elif kind == "balanced":
        N, d = case["N"], case["d"]
        unit = lambda t: t / t.norm(dim=-1, keepdim=True)
        p.update(Q=unit(rnd(B, H, N, d)), K=unit(rnd(B, H, N, d)), x=_chain(g, B, N, dev), V=rnd(B, H, N, d),
                 alpha=-1.0 + 0.3 * rnd(H), r=10.0 + rnd(H))
        const.update(eps=_trunk_eps(H, dev), mask=_mask(case, N, dev))
        s["grad"] = [rnd(B, H, N, 3), rnd(B, H, N, d)]
    elif kind == "block":
        N, C = case["N"], case["C"]
        lin = torch.nn.Linear
        block = SimpleNamespace(
            n_heads=H, feature_transport=True, ln_sink=torch.nn.LayerNorm(C).to(dev),
            w_q_sink=lin(C, C, bias=False, device=dev), w_k_sink=lin(C, C, bias=False, device=dev),
            w_v_sink=lin(C, C, bias=False, device=dev), w_o_sink=lin(C, C, bias=False, device=dev),
            ln_gate=torch.nn.LayerNorm(C).to(dev), w_gate=lin(C, 1, device=dev),
            alpha_h=torch.nn.Parameter(torch.full((H,), -1.0, device=dev)),
            r_h=torch.nn.Parameter(torch.full((H,), 10.0, device=dev)), eps=_trunk_eps(H, dev),
            lambda_h_raw=torch.nn.Parameter(torch.zeros(H, device=dev)))
        with torch.no_grad():
            for m in (block.w_q_sink, block.w_k_sink, block.w_v_sink, block.w_o_sink, block.w_gate):
                m.weight.copy_(rnd(*m.weight.shape, scale=C ** -0.5))
            block.w_gate.bias.copy_(rnd(1, scale=0.1))
            for ln in (block.ln_sink, block.ln_gate):
                ln.weight.copy_(1 + 0.1 * rnd(C))
                ln.bias.copy_(0.1 * rnd(C))
            block.lambda_h_raw.copy_(0.3 * rnd(H))
        s["block"] = block
        p.update(h=rnd(B, N, C), x=_chain(g, B, N, dev))
        for n, t in _block_params(block).items():
            p[n] = t
        const["mask"] = _mask(case, N, dev)
        s["grad"] = [rnd(B, N, C), rnd(B, N, 3)]
    elif kind == "dense":
        N, d = case["N"], case["d"]
        q, k = rnd(B, H, N, d), rnd(B, H, N, d)
        cost = -(q @ k.transpose(-1, -2).contiguous()) / math.sqrt(d) + 0.3 * torch.rand(B, H, N, N, generator=g,
                                                                                          device=dev)
        p.update(C=cost.contiguous(), V=rnd(B, H, N, d), G=rnd(B, H, N, d), x=_chain(g, B, N, dev))
        p["log_mu"], p["log_nu"] = _marginals(case, g, dev)
        const.update(eps=torch.linspace(0.5, 1.5, H, device=dev), mask=_mask(case, N, dev))
        s["grad"] = [rnd(B, N, H * d), rnd(B, H, N, 3, scale=0.3)]
    elif kind == "diffusion":
        N, d = case["N"], case["d"]
        p.update(Q=rnd(B, H, N, d, dtype=dt), K=rnd(B, H, N, d, dtype=dt), V=rnd(B, H, N, d, dtype=dt))
        if case["gate"]:
            p["G"] = rnd(B, H, N, d, dtype=dt)
        if case["bias"] == "dense":
            p["bias"] = rnd(B, H, N, N, dtype=dt)
        else:
            i = torch.arange(N, device=dev)
            rel = (i[:, None] - i[None, :]).clamp(-32, 32) + 32
            const["bins"] = rel[None].expand(B, N, N).to(torch.int32).contiguous()
            p["pos_weight"] = rnd(H, BINS, scale=0.5)
        const["mask"] = _mask(case, N, dev)
        s["grad"] = [rnd(B, H, N, d, dtype=dt)]
    elif kind == "window":
        M, d = case["M"], case["d"]
        p.update(Q=rnd(B, H, M, d, dtype=dt), K=rnd(B, H, M, d, dtype=dt), V=rnd(B, H, M, d, dtype=dt))
        if case["bias"]:
            p["bias"] = rnd((M + 31) // 32, H, 32, 128, dtype=dt)
        const["mask"] = _mask(case, M, dev)
        s["grad"] = [rnd(B, H, M, d, dtype=dt)]
    else:
        M, d = case["M"], case["d"]
        N = M // ATOMS
        p.update(Qa=rnd(B, H, M, d, dtype=dt), Kt=rnd(B, H, N, d, dtype=dt), Vt=rnd(B, H, N, d, dtype=dt),
                 Qt=rnd(B, H, N, d, dtype=dt), Ka=rnd(B, H, M, d, dtype=dt), Va=rnd(B, H, M, d, dtype=dt))
        r = torch.randint(-10, 11, (B, N // 2), generator=g, device=dev)  # 14 to 34 atoms a token
        counts = torch.full((B, N), ATOMS, device=dev)
        counts[:, 0:2 * (N // 2):2] += r
        counts[:, 1:2 * (N // 2):2] -= r
        const["counts"] = counts.to(torch.int32)
        const["starts"] = (torch.cumsum(counts, 1) - counts).to(torch.int32)
        s["grad"] = [rnd(B, H, M, d, dtype=dt), rnd(B, H, N, d, dtype=dt)]
    if case.get("train", True):
        for t in p.values():
            t.requires_grad_(True)
    return s


def _trunk_eps(H, dev):
    """The trunk's regularisation: 0.5, 1, 2 and 4 over the quarters of the heads."""
    return torch.tensor([0.5, 1.0, 2.0, 4.0], device=dev)[torch.arange(H, device=dev) * 4 // H]


def _block_params(b):
    return dict(ln_sink_w=b.ln_sink.weight, ln_sink_b=b.ln_sink.bias, w_q=b.w_q_sink.weight, w_k=b.w_k_sink.weight,
                w_v=b.w_v_sink.weight, w_o=b.w_o_sink.weight, alpha=b.alpha_h, r=b.r_h, ln_gate_w=b.ln_gate.weight,
                ln_gate_b=b.ln_gate.bias, w_gate=b.w_gate.weight, b_gate=b.w_gate.bias, lam=b.lambda_h_raw)


def run(state):
    import deepfold_amd as df

    case, p, c = state["case"], state["p"], state["const"]
    kind, train = case["kind"], case.get("train", True)
    if not train:
        with torch.no_grad():
            return dict(zip(_names(case), _forward(df, kind, case, p, c, state)))
    out = _forward(df, kind, case, p, c, state)
    loss = [out[i] for i in _loss(case)]
    grads = torch.autograd.grad(loss, list(p.values()), state["grad"])
    res = dict(zip(_names(case), out))
    res.update({"d_" + n: t for n, t in zip(p, grads)})
    return {n: t.detach() for n, t in res.items()}


def _names(case):
    return {"uot": ("o", "xc", "log_u", "log_v"), "unrolled": ("o", "xc", "log_u", "log_v"), "balanced": ("xc", "hc"),
            "block": ("h", "x"), "dense": ("log_u", "log_v", "o", "T", "xc"), "diffusion": ("o",), "window": ("o",),
            "cross": ("atoms", "tokens")}[case["kind"]]


def _loss(case):
    """The outputs that the loss reaches."""
    if case["kind"] in ("uot", "unrolled"):
        return (0, 1) if case["full"] else (0,)
    return {"balanced": (0, 1), "block": (0, 1), "dense": (2, 4), "diffusion": (0,), "window": (0,),
            "cross": (0, 1)}[case["kind"]]


def _forward(df, kind, case, p, c, state):
    if kind in ("uot", "unrolled"):
        x, pw, wd = p.get("x", c.get("x")), p.get("pos_weight", c.get("pos_weight")), p.get("w_dist")
        if kind == "unrolled":
            return df.flash_sinkhorn(p["Q"], p["K"], p["V"], x, pw, c["bins"], c["eps"], wd, p["log_mu"], p["log_nu"],
                                     K_iter=case["K"], r_0=R0, mask=c["mask"])
        kw = dict(ift_solver="cg", ift_iters=case["iters"]) if case["iters"] else {}
        return df.flash_sinkhorn_attn(p["Q"], p["K"], p["V"], p["G"], x, pw, c["bins"], c["eps"], wd, p["log_mu"],
                                      p["log_nu"], K_iter=case["K"], r_0=R0, mask=c["mask"], **kw)
    if kind == "balanced":
        return df.balanced_sinkhorn_transport_dual(p["Q"], p["K"], p["x"], p["V"], c["eps"], p["alpha"], p["r"],
                                                   K_iter=case["K"], mask=c["mask"])
    if kind == "block":
        return df.token_ot_transport_step(state["block"], p["h"], p["x"], c["mask"], K_iter=case["K"])
    if kind == "dense":
        lu, lv = df.sinkhorn_solve(p["C"], p["log_mu"], p["log_nu"], c["eps"], K=case["K"], mask=c["mask"])
        return (lu, lv) + df.compute_transport_output(p["V"], p["G"], lu, lv, p["C"], c["eps"], p["x"], c["mask"])
    if kind == "diffusion":
        return (df.flash_diffusion_attn(p["Q"], p["K"], p["V"], p.get("pos_weight"), c.get("bins"), c["mask"],
                                        pair_bias=p.get("bias"), gate=p.get("G")),)
    if kind == "window":
        return (df.flash_atom_attn(p["Q"], p["K"], p["V"], c["mask"], window_bias=p.get("bias")),)
    return (df.token_to_atom_attn(p["Qa"], p["Kt"], p["Vt"]),
            df.atom_to_token_attn(p["Qt"], p["Ka"], p["Va"], c["starts"], c["counts"]))


def work(case):
    """Inputs read once, outputs written once; products, and two operations an element and half-iteration."""
    kind, B, H = case["kind"], case["B"], case["H"]
    e = 2 if case.get("dtype") == "bf16" else 4
    train = case.get("train", True)
    n = case.get("N", case.get("M"))
    E = H * sum(k * k for k in _lengths(case, n))
    if kind in ("uot", "unrolled"):
        d, K = case["d"], case["K"]
        rows = B * H * n
        nbytes = rows * (4 * d * e + 4 * d + 4 * 7)
        flops = E * (4 * d + 6 + 4 * K)
        if train:
            nbytes += rows * (4 * d + 4 * d * e + 8)
            flops += E * (8 * d + 4 * (case.get("iters") or K))
        if case["full"]:
            nbytes += 4 * B * n * n
        return {"bytes": nbytes, "flops": flops}
    if kind == "balanced":
        d = case["d"]
        return {"bytes": 4 * B * H * n * (8 * d + 6), "flops": E * (12 * d + 18 + 8 * case["K"])}
    if kind == "block":
        C, d = case["C"], case["C"] // H
        rows = B * n
        return {"bytes": 4 * (rows * 4 * C + 8 * C * C),
                "flops": 24 * rows * C * C + E * (12 * d + 18 + 8 * case["K"])}
    if kind == "dense":
        d = case["d"]
        full = B * H * n * n
        return {"bytes": 4 * (3 * full + B * H * n * (6 * d + 10)), "flops": E * (6 * d + 12 * case["K"])}
    d = case["d"]
    if kind == "diffusion":
        rows = B * H * n
        big = B * H * n * n * e if case["bias"] == "dense" else 4 * B * n * n
        t = rows * d * e * (4 + (1 if case["gate"] else 0))
        if train:
            t += rows * d * e * (4 + (1 if case["gate"] else 0))
            big *= 2 if case["bias"] == "dense" else 1
        return {"bytes": big + t, "flops": E * d * (14 if train else 4)}
    if kind == "window":
        rows = B * H * n
        big = ((n + 31) // 32) * H * 32 * 128 * e if case["bias"] else 0
        return {"bytes": (2 if train else 1) * (big + 4 * rows * d * e), "flops": rows * 128 * d * (14 if train else 4)}
    N = n // ATOMS
    t = B * H * d * e * (2 * n + 2 * N + 2 * N + 2 * n)
    return {"bytes": (2 if train else 1) * t, "flops": B * H * n * (N + 1) * d * (14 if train else 4)}


def tolerance(case):
    """About four times the largest error against float64 of any output over these ranges: 1.5e-5 in fp32 (the
    gradient of a scalar bias), in bf16 3.1e-3, and 4.3e-3 for a bias table's gradient summed from bf16 terms."""
    if case.get("dtype") != "bf16":
        return {"rel": 6e-5}
    return {"rel": 1.2e-2} if case["kind"] in ("uot", "unrolled") else {"rel": 1.7e-2}


# ---------------------------------------------------------------------------------------
# The same passes in float64 torch.


def exact(case, seed):
    s = prepare(case, seed)
    kind, train = case["kind"], case.get("train", True)
    p = {n: t.detach().double() for n, t in s["p"].items()}
    c = {n: (t.double() if t is not None and t.is_floating_point() else t) for n, t in s["const"].items()}
    grad = [t.double() for t in s["grad"]]
    if kind == "uot":
        return _exact_uot(case, p, c, grad)
    if train:
        for t in p.values():
            t.requires_grad_(True)
    out = {"unrolled": _exact_unrolled, "balanced": _exact_balanced, "block": _exact_block, "dense": _exact_dense,
           "diffusion": _exact_diffusion, "window": _exact_window, "cross": _exact_cross}[kind](case, p, c)
    res = dict(zip(_names(case), out))
    if train:
        grads = torch.autograd.grad([out[i] for i in _loss(case)], list(p.values()), grad)
        res.update({"d_" + n: t for n, t in zip(p, grads)})
    return {n: t.detach() for n, t in res.items()}


def _distance(x):
    """(n, n) distances and their gradient, zero on the diagonal."""
    diff = x[..., :, None, :] - x[..., None, :, :]
    return diff.pow(2).sum(-1).clamp(min=1e-16).sqrt()


def _t(a):
    return a.transpose(-1, -2).contiguous()


def _exact_uot(case, p, c, grad):
    """Sinkhorn iterations, then the implicit gradient: one group of heads of one sample at a time."""
    B, H, N, d, K = case["B"], case["H"], case["N"], case["d"], case["K"]
    train, full = case["train"], case["full"]
    z = lambda *sh: torch.zeros(*sh, dtype=torch.float64, device=p["Q"].device)
    res = dict(o=z(B, N, H * d), xc=z(B, H, N, 3), log_u=z(B, H, N), log_v=z(B, H, N))
    if train:
        res.update({"d_" + n: torch.zeros_like(t) for n, t in p.items()})
    xs = p.get("x", c.get("x"))
    for b, n in enumerate(_lengths(case, N)):
        x = xs[b, :n]
        group = max(1, min(H, (1 << 26) // (n * n)))
        dist = _distance(x) if full else None
        diff = x[:, None, :] - x[None, :, :] if full else None
        for h0 in range(0, H, group):
            hs = slice(h0, min(H, h0 + group))
            q, k, v, gt = (p[m][b, hs, :n] for m in ("Q", "K", "V", "G"))
            eps = c["eps"][hs, None, None]
            kap = (1.0 / (1.0 + c["eps"][hs]))[:, None]
            cost = -(q @ _t(k)) / math.sqrt(d)
            if full:
                w = p["w_dist"][hs, None, None]
                bins = c["bins"][b, :n, :n].long()
                cost = cost + w * (dist / (R0 + dist)) + p["pos_weight"][hs][:, bins]
            L = -cost / eps
            mu, nu = p["log_mu"][b, hs, :n], p["log_nu"][b, hs, :n]
            u, vv = torch.zeros_like(mu), torch.zeros_like(nu)
            for _ in range(K):
                u = kap * (mu - torch.logsumexp(L + vv[:, None, :], -1))
                vv = kap * (nu - torch.logsumexp(L + u[:, :, None], -2))
            lz = torch.logsumexp(L + vv[:, None, :], -1)
            T = torch.exp(L + vv[:, None, :] - lz[:, :, None])
            oa, xc = T @ v, T @ x
            sg = torch.sigmoid(gt)
            o4 = res["o"].view(B, N, H, d)
            o4[b, :n, hs] = (sg * oa).transpose(0, 1)
            res["xc"][b, hs, :n], res["log_u"][b, hs, :n], res["log_v"][b, hs, :n] = xc, u, vv
            if not train:
                continue
            go = grad[0].view(B, N, H, d)[b, :n, hs].transpose(0, 1)
            gx = grad[1][b, hs, :n] if full else torch.zeros_like(xc)
            gO = sg * go
            res["d_G"][b, hs, :n] = sg * (1 - sg) * oa * go
            D = (gO * oa).sum(-1) + (gx * xc).sum(-1)
            gls = T * (gO @ _t(v) + gx @ _t(x) - D[:, :, None])
            g_v = gls.sum(1)
            Tt = _t(T)
            res["d_V"][b, hs, :n] = Tt @ gO
            S_row = T
            S_col = torch.softmax(L + u[:, :, None], dim=1)
            kap1 = kap
            if case["iters"]:
                # (I - kappa^2 S_row^T S_col) z_v = g_v on its symmetric form, solved by CG
                P = torch.exp(u[:, :, None] + L + vv[:, None, :])
                r, cs = P.sum(2), P.sum(1)
                W = P / r.sqrt()[:, :, None] / cs.sqrt()[:, None, :]
                Wt = _t(W)
                rhs = g_v / cs.sqrt()
                y, res_, q_ = torch.zeros_like(rhs), rhs.clone(), rhs.clone()
                rr = (res_ * res_).sum(-1, keepdim=True)
                for _ in range(case["iters"]):
                    Aq = q_ - kap1 ** 2 * (Wt @ (W @ q_[:, :, None]))[:, :, 0]
                    den = (q_ * Aq).sum(-1, keepdim=True)
                    al = torch.where(den > 0, rr / den.clamp(min=1e-300), torch.zeros_like(den))
                    y, res_ = y + al * q_, res_ - al * Aq
                    new = (res_ * res_).sum(-1, keepdim=True)
                    q_ = res_ + torch.where(rr > 0, new / rr.clamp(min=1e-300), torch.zeros_like(rr)) * q_
                    rr = new
                z_v = cs.sqrt() * y
                z_u = kap1 * (S_col @ z_v[:, :, None])[:, :, 0]
            else:
                z_v = g_v.clone()
                for _ in range(K):
                    z_u = kap1 * (S_col @ z_v[:, :, None])[:, :, 0]
                    z_v = g_v + kap1 * (Tt @ z_u[:, :, None])[:, :, 0]
            dC = -gls / eps - (kap1[:, :, None] / eps) * (z_u[:, :, None] * S_row + z_v[:, None, :] * S_col)
            res["d_Q"][b, hs, :n] = -(dC @ k) / math.sqrt(d)
            res["d_K"][b, hs, :n] = -(_t(dC) @ q) / math.sqrt(d)
            res["d_log_mu"][b, hs, :n] = kap1 * z_u
            res["d_log_nu"][b, hs, :n] = kap1 * z_v
            if full:
                f = dC * (w * R0 / (R0 + dist) ** 2) / dist
                fs = f.sum(0)
                res["d_x"][b, :n] += (Tt @ gx).sum(0) + (fs[:, :, None] * diff).sum(1) - (fs[:, :, None] * diff).sum(0)
                res["d_w_dist"][hs] += (dC * (dist / (R0 + dist))).sum((1, 2))
                for i in range(dC.shape[0]):
                    res["d_pos_weight"][h0 + i] += torch.zeros(BINS, dtype=torch.float64, device=x.device).index_add_(
                        0, bins.reshape(-1), dC[i].reshape(-1))
    return res


def _pad(t, n, dim):
    """t with zeros after its valid tokens, up to n of them."""
    sh = list(t.shape)
    sh[dim] = n - sh[dim]
    return torch.cat([t, torch.zeros(sh, dtype=t.dtype, device=t.device)], dim) if sh[dim] else t


def _exact_unrolled(case, p, c):
    B, H, N, d = case["B"], case["H"], case["N"], case["d"]
    outs = []
    xs, kap = p.get("x", c.get("x")), (1.0 / (1.0 + c["eps"]))[:, None]
    for b, n in enumerate(_lengths(case, N)):
        q, k, v, x = p["Q"][b, :, :n], p["K"][b, :, :n], p["V"][b, :, :n], xs[b, :n]
        cost = -(q @ _t(k)) / math.sqrt(d)
        if case["full"]:
            dist = _distance(x)
            cost = cost + p["w_dist"][:, None, None] * (dist / (R0 + dist))
            cost = cost + p["pos_weight"][:, c["bins"][b, :n, :n].long()]
        L = -cost / c["eps"][:, None, None]
        mu, nu = p["log_mu"][b, :, :n], p["log_nu"][b, :, :n]
        u, w = torch.zeros_like(mu), torch.zeros_like(nu)
        for _ in range(case["K"]):
            u = kap * (mu - torch.logsumexp(L + w[:, None, :], -1))
            w = kap * (nu - torch.logsumexp(L + u[:, :, None], -2))
        T = torch.softmax(L + w[:, None, :], -1)
        outs.append([_pad(t, N, 1) for t in (T @ v, T @ x, u, w)])
    return tuple(torch.stack([o[i] for o in outs]) for i in range(4))


def _balanced(case, q, k, x, v, eps, alpha, r, n):
    w = torch.sigmoid(alpha)[:, None, None]
    dist = _distance(x)
    L = -((1 - w) * (1 - q @ _t(k)) + w * (dist / (r.abs().clamp(min=0.1)[:, None, None] + dist))) / eps[:, None, None]
    lm = -math.log(n)
    u = torch.zeros(q.shape[0], n, dtype=q.dtype, device=q.device)
    for _ in range(case["K"]):
        vv = lm - torch.logsumexp(L + u[:, :, None], -2)
        u = lm - torch.logsumexp(L + vv[:, None, :], -1)
    T = torch.softmax(L + vv[:, None, :], -1)
    return T @ x, T @ v


def _exact_balanced(case, p, c):
    N, outs = case["N"], []
    for b, n in enumerate(_lengths(case, N)):
        o = _balanced(case, p["Q"][b, :, :n], p["K"][b, :, :n], p["x"][b, :n], p["V"][b, :, :n], c["eps"], p["alpha"],
                      p["r"], n)
        outs.append([_pad(t, N, 1) for t in o])
    return tuple(torch.stack([o[i] for o in outs]) for i in range(2))


def _exact_block(case, p, c):
    B, H, N, C = case["B"], case["H"], case["N"], case["C"]
    norm = torch.nn.functional.layer_norm
    h, x, eps = p["h"], p["x"], _trunk_eps(H, p["h"].device).double()
    hs = norm(h, (C,), p["ln_sink_w"], p["ln_sink_b"], 1e-5)
    heads = lambda w: (hs @ _t(w)).view(B, N, H, C // H).transpose(1, 2)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True).clamp(min=1e-12)
    q, k, v = unit(heads(p["w_q"])), unit(heads(p["w_k"])), heads(p["w_v"])
    m = torch.ones(B, N, dtype=h.dtype, device=h.device) if c["mask"] is None else c["mask"]
    xc, hc = [], []
    for b, n in enumerate(_lengths(case, N)):
        o = _balanced(case, q[b, :, :n], k[b, :, :n], x[b, :n], v[b, :, :n], eps, p["alpha"], p["r"], n)
        xc.append(_pad(o[0], N, 1))
        hc.append(_pad(o[1], N, 1))
    xc, hc = torch.stack(xc), torch.stack(hc)
    h = h + (hc.transpose(1, 2).reshape(B, N, C) @ _t(p["w_o"])) * m[:, :, None]
    gate = torch.sigmoid(norm(h, (C,), p["ln_gate_w"], p["ln_gate_b"], 1e-5) @ _t(p["w_gate"]) + p["b_gate"])
    lam = (torch.tanh(p["lam"]) / H)[None, :, None, None]
    return h, x + m[:, :, None] * gate * (lam * (xc - x[:, None])).sum(1)


def _exact_dense(case, p, c):
    B, H, N, d = case["B"], case["H"], case["N"], case["d"]
    outs, kap = [], (1.0 / (1.0 + c["eps"]))[:, None]
    for b, n in enumerate(_lengths(case, N)):
        L = -p["C"][b, :, :n, :n] / c["eps"][:, None, None]
        mu, nu = p["log_mu"][b, :, :n], p["log_nu"][b, :, :n]
        u, w = torch.zeros_like(mu), torch.zeros_like(nu)
        for _ in range(case["K"]):
            u = kap * (mu - torch.logsumexp(L + w[:, None, :], -1))
            w = kap * (nu - torch.logsumexp(L + u[:, :, None], -2))
        s = u[:, :, None] + L + w[:, None, :]
        T = torch.exp(s - s.amax(-1, keepdim=True))
        T = T / (T.sum(-1, keepdim=True) + 1e-6)
        o = torch.sigmoid(p["G"][b, :, :n]) * (T @ p["V"][b, :, :n])
        outs.append([_pad(u, N, 1), _pad(w, N, 1), _pad(o.transpose(0, 1).reshape(n, H * d), N, 0),
                     _pad(_pad(T, N, 1), N, 2), _pad(T @ p["x"][b, :n], N, 1)])
    return tuple(torch.stack([o[i] for o in outs]) for i in range(5))


def _exact_diffusion(case, p, c):
    N, d = case["N"], case["d"]
    s = (p["Q"] @ _t(p["K"])) / math.sqrt(d)
    if "bias" in p:
        s = s + p["bias"]
    else:
        s = s + p["pos_weight"][:, c["bins"].long()].transpose(0, 1)
    if c["mask"] is not None:
        s = s.masked_fill(c["mask"][:, None, None, :] == 0, float("-inf"))
    o = torch.softmax(s, -1) @ p["V"]
    if c["mask"] is not None:
        o = o * c["mask"][:, None, :, None]
    return (o * torch.sigmoid(p["G"]) if "G" in p else o,)


def _exact_window(case, p, c):
    """Window w: queries [32w, 32w + 32) and keys [32w - 48, 32w + 80) of the sequence."""
    B, H, M, d = case["B"], case["H"], case["M"], case["d"]
    W = (M + 31) // 32
    dev = p["Q"].device
    keys = torch.arange(W, device=dev)[:, None] * 32 - 48 + torch.arange(128, device=dev)
    ok = ((keys >= 0) & (keys < M))[None].expand(B, W, 128)
    at = keys.clamp(0, M - 1)
    if c["mask"] is not None:
        ok = ok & (c["mask"][:, at] > 0)
    q = _pad(p["Q"], W * 32, 2).view(B, H, W, 32, d)
    k, v = p["K"][:, :, at], p["V"][:, :, at]
    s = (q @ _t(k)) / math.sqrt(d)
    if "bias" in p:
        s = s + p["bias"].transpose(0, 1)[None]
    s = s.masked_fill(~ok[:, None, :, None, :], -1e30)
    o = (torch.softmax(s, -1) @ v).reshape(B, H, W * 32, d)[:, :, :M]
    return (o if c["mask"] is None else o * c["mask"][:, None, :, None],)


def _exact_cross(case, p, c):
    M, d = case["M"], case["d"]
    atoms = torch.softmax((p["Qa"] @ _t(p["Kt"])) / math.sqrt(d), -1) @ p["Vt"]
    j = torch.arange(M, device=p["Qa"].device)
    st, ct = c["starts"].long()[:, :, None], c["counts"].long()[:, :, None]
    s = (p["Qt"] @ _t(p["Ka"])) / math.sqrt(d)
    s = s.masked_fill(~((j >= st) & (j < st + ct))[:, None], float("-inf"))
    return atoms, torch.softmax(s, -1) @ p["Va"]
