"""The measured cases: what a program that uses mamba_hip has it do.

``listed()`` are twelve calls through the package's public entry points,
``draw()`` more of the same ranges.  ``prepare`` makes what the program has in
hand before the call (inputs, weights, caches, a captured decode step), ``run``
is one pass, ``exact`` the same result in 64 bits by plain torch.

Tolerances come from the data types.  ``tests/`` holds the finer comparisons.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "burn-mamba_amd"))

import mamba_hip  # noqa: E402

DEV = "cuda"
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
# how many layers the decode cases step: more weights than the last-level cache
# holds at the Mamba-2 sizes, few enough that roundings do not travel far
LAYERS = 8


# ------------------------------------------------------------------ the cases --

def listed():
    return [
        # The SSD alone in the reference's default float, at the size of its
        # CPU-runnable check: two short sequences, few heads.
        dict(name="ssd2_small_f32", kind="ssd2", dtype="f32", b=2, l=512, h=8, p=64, g=1, n=64, chunk=64, h0=False),
        # The SSD of a Mamba-2 2.7B layer in a batched prefill.
        dict(name="ssd2_prefill", kind="ssd2", dtype="bf16", b=8, l=4096, h=80, p=64, g=1, n=128, chunk=256, h0=False),
        # One prompt alone, of odd length, that continues a cached state.
        dict(name="ssd2_prompt", kind="ssd2", dtype="bf16", b=1, l=3001, h=80, p=64, g=1, n=128, chunk=256, h0=True),
        # A training step through the SSD: forward, then every gradient.
        dict(name="ssd2_train", kind="ssd2_train", dtype="bf16", b=2, l=2048, h=80, p=64, g=1, n=128, chunk=256),
        # The whole Mamba-2 block over two prompts of odd length (serving).
        dict(name="mamba2_block", kind="mamba2_block", b=2, l=1021, d_model=2560, n=128),
        # One decode step at the headline batch, replayed from a graph as a
        # serving loop does.
        dict(name="mamba2_decode", kind="mamba2_decode", b=64, d_model=2560, n=128),
        # One decode step for a single user: latency of small launches.
        dict(name="mamba3_decode", kind="mamba3_decode", b=1, d_model=1024, n=128, mimo=4),
        # The Mamba-1 2.8B selective scan, batched.
        dict(name="mamba1_scan", kind="mamba1_scan", b=8, d=5120, l=2048, n=16),
        # The Mamba-1 block at the reference's own benchmark shape: many small launches.
        dict(name="mamba1_block", kind="mamba1_block", b=2, l=256, d_model=256, n=16),
        # A batched Mamba-3 prefill with long sequences and MIMO rank 4.
        dict(name="mamba3_prefill", kind="mamba3_prefill", b=4, l=8192, d_model=1024, n=128, mimo=4),
        # The Mamba-3 block in f32 at the reference's own benchmark shape.
        dict(name="mamba3_block_f32", kind="mamba3_block", b=2, l=256, d_model=256, n=64, mimo=4),
        # A training step through the Mamba-3 SSD in the reference's default float.
        dict(name="mamba3_train", kind="mamba3_train", dtype="f32", b=2, l=4096, h=32, p=64, n=128, mimo=4, chunk=64),
    ]


def _spread(rng, lo, hi):
    """A whole number of lo..hi, spread evenly over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["ssd2_f32", "ssd2_bf16", "ssd2_train", "mamba2_block", "mamba2_decode", "mamba3_decode",
                       "mamba1_scan", "mamba1_block", "mamba3_prefill", "mamba3_block", "mamba3_train"])
    if kind == "ssd2_f32":
        return dict(kind="ssd2", dtype="f32", b=rng.randint(1, 4), l=_spread(rng, 64, 1024), h=rng.choice([4, 8, 16, 24]),
                    p=rng.choice([32, 64, 64, 128]), g=rng.choice([1, 1, 2]), n=rng.choice([32, 64, 64, 128]),
                    chunk=rng.choice([64, 128, 256]), h0=rng.random() < 0.5)
    if kind == "ssd2_bf16":
        return dict(kind="ssd2", dtype="bf16", b=rng.randint(1, 8), l=_spread(rng, 256, 4096),
                    h=rng.choice([24, 32, 48, 64, 80]), p=64, g=rng.choice([1, 1, 1, 2]), n=rng.choice([64, 128, 128]),
                    chunk=rng.choice([128, 256]), h0=rng.random() < 0.5)
    if kind == "ssd2_train":
        return dict(kind=kind, dtype=rng.choice(["bf16", "f32"]), b=rng.randint(1, 2), l=_spread(rng, 256, 2048),
                    h=rng.choice([24, 48, 80]), p=64, g=1, n=rng.choice([64, 128, 128]), chunk=rng.choice([128, 256]))
    if kind == "mamba2_block":
        return dict(kind=kind, b=rng.randint(1, 4), l=_spread(rng, 64, 2048), d_model=rng.choice([768, 1024, 1536, 2560]),
                    n=rng.choice([64, 128, 128]))
    if kind == "mamba2_decode":
        return dict(kind=kind, b=_spread(rng, 1, 128), d_model=rng.choice([1024, 2560]), n=128)
    if kind == "mamba3_decode":
        return dict(kind=kind, b=_spread(rng, 1, 128), d_model=rng.choice([1024, 2048]), n=128, mimo=rng.choice([1, 4]))
    if kind == "mamba1_scan":
        return dict(kind=kind, b=rng.randint(1, 8), d=rng.choice([1536, 2560, 5120]), l=_spread(rng, 256, 2048), n=16)
    if kind == "mamba1_block":
        return dict(kind=kind, b=rng.randint(1, 4), l=_spread(rng, 32, 1024), d_model=rng.choice([256, 512, 1024]), n=16)
    if kind == "mamba3_prefill":
        return dict(kind=kind, b=rng.randint(1, 4), l=_spread(rng, 512, 8192), d_model=rng.choice([512, 1024]), n=128,
                    mimo=rng.choice([1, 2, 4]))
    if kind == "mamba3_block":
        return dict(kind=kind, b=rng.randint(1, 4), l=_spread(rng, 32, 512), d_model=rng.choice([256, 512]),
                    n=rng.choice([64, 128]), mimo=rng.choice([1, 4]))
    # long sequences at the full state, the reference benchmark's block at its own
    n = rng.choice([64, 128, 128])
    return dict(kind="mamba3_train", dtype=rng.choice(["bf16", "f32"]), b=rng.randint(1, 2),
                l=_spread(rng, 128, 2048 if n == 128 else 512), h=rng.choice([8, 16, 32]), p=64, n=n,
                mimo=rng.choice([1, 4]), chunk=rng.choice([64, 128]))


# --------------------------------------------------------------------- inputs --

def _dtype(case):
    return BF16 if case.get("dtype", "bf16") == "bf16" else F32


class _Rand:
    """Seeded values on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.gen, device=DEV) * std

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.gen, device=DEV) * (hi - lo) + lo

    def dt(self, h, *shape):
        """dt = softplus(N(0, 1) + b_h) around the reference's dt init (1e-3 .. 0.1)."""
        t = torch.exp(self.uniform(math.log(1e-3), math.log(0.1), h))
        return F.softplus(self.normal(*shape, h) + t + torch.log(-torch.expm1(-t)))


def _ssd2_inputs(case, seed):
    r, io = _Rand(seed), _dtype(case)
    b, l, h, p, g, n = (case[k] for k in "blhpgn")
    t = dict(x=r.normal(b, l, h, p).to(io), dt=r.dt(h, b, l), A=-torch.exp(r.uniform(0.0, math.log(16.0), h)),
             B=r.normal(b, l, g, n, std=n ** -0.5).to(io), C=r.normal(b, l, g, n, std=n ** -0.5).to(io), D=r.normal(h))
    t["h0"] = r.normal(b, h, p, n, std=0.1) if case.get("h0", True) else None
    if case["kind"] == "ssd2_train":
        t["dy"], t["dhT"] = r.normal(b, l, h, p).to(io), r.normal(b, h, p, n)
    return t


def _mamba3_train_inputs(case, seed):
    r, io = _Rand(seed), _dtype(case)
    b, l, h, p, n, m = (case[k] for k in ("b", "l", "h", "p", "n", "mimo"))
    dt, A = r.dt(h, b, l), -torch.exp(r.uniform(0.0, math.log(16.0), h))
    lam = torch.sigmoid(r.normal(b, l, h))
    gamma = lam * dt
    scale = gamma.clone()
    scale[:, :-1] += (1 - lam[:, 1:]) * dt[:, 1:]
    return dict(v=r.normal(b, l, m, h, p).to(io), da=dt * A, B=r.normal(b, l, m, h, n, std=n ** -0.5).to(io),
                C=r.normal(b, l, m, h, n, std=n ** -0.5).to(io), gamma=gamma, scale=scale,
                h0=r.normal(b, h, p, n, std=0.1), dy=r.normal(b, l, m, h, p).to(io), dhT=r.normal(b, h, p, n))


def _mamba1_scan_inputs(case, seed):
    r = _Rand(seed)
    b, d, l, n = (case[k] for k in "bdln")
    return dict(u=r.normal(b, d, l), delta=F.softplus(r.normal(b, d, l) - 4.0),
                A=-torch.arange(1.0, n + 1, device=DEV).repeat(d, 1), B=r.normal(b, n, l), C=r.normal(b, n, l),
                D=torch.ones(d, device=DEV), z=r.normal(b, d, l))


def _block(case, seed):
    """The block of a case, its input, and the program's generator."""
    r = _Rand(seed)
    if case["kind"] == "mamba1_block":
        m = mamba_hip.Mamba1Config(case["d_model"], state_rank=case["n"]).init(DEV, r.gen)
    elif case["kind"] == "mamba2_block":
        m = mamba_hip.Mamba2Config(case["d_model"], state_rank=case["n"]).init(DEV, BF16, r.gen)
    else:
        io = BF16 if case["kind"] == "mamba3_prefill" else F32
        m = mamba_hip.Mamba3Config(case["d_model"], state_rank=case["n"], mimo_rank=case["mimo"]).init(DEV, io, r.gen)
    x = r.normal(case["b"], case["l"], case["d_model"])
    return m, x if case["kind"] in ("mamba1_block", "mamba3_block") else x.to(BF16)


def _stack(case, seed):
    """The stack of a decode case, its caches in mid-conversation and the token's row."""
    r = _Rand(seed)
    b = case["b"]
    if case["kind"] == "mamba2_decode":
        cfg = mamba_hip.Mamba2Config(case["d_model"], state_rank=case["n"])
        stack = mamba_hip.Mamba2Stack.init(cfg, LAYERS, DEV, BF16, r.gen)
        caches = [mamba_hip.Mamba2Cache(r.normal(b, cfg.conv_dim, cfg.conv_kernel),
                                        r.normal(b, cfg.nheads, cfg.per_head_dim, cfg.state_rank, std=0.1))
                  for _ in range(LAYERS)]
    else:
        cfg = mamba_hip.Mamba3Config(case["d_model"], state_rank=case["n"], mimo_rank=case["mimo"])
        stack = mamba_hip.Mamba3Stack.init(cfg, LAYERS, DEV, BF16, r.gen)
        H, P, N = cfg.nheads, cfg.per_head_dim, cfg.state_rank
        caches = [mamba_hip.Mamba3Cache(r.normal(b, H, P, N, std=0.1), r.normal(b, cfg.mimo_rank, H, N),
                                        r.normal(b, H, P), r.uniform(-3.0, 3.0, b, H, cfg.num_rope_angles))
                  for _ in range(LAYERS)]
    return stack, caches, r.normal(b, case["d_model"])


def _tensors(cache):
    """The tensors of a decode cache that a program reads back.  Mamba-3's
    angle is left out: it is kept modulo 2 pi, so that equal angles can be
    numbers 2 pi apart, and K is B rotated by it."""
    if isinstance(cache, mamba_hip.Mamba2Cache):
        return dict(conv=cache.conv_bvk, ssm=cache.ssm_bhpr)
    if isinstance(cache, mamba_hip.Mamba1Cache):
        return dict(conv=cache.conv_bik, ssm=cache.ssm_bir)
    return dict(ssm=cache.ssm_bhpr, k=cache.k_state_bmhr, v=cache.v_state_bhp)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "ssd2":
        return dict(case=case, **_ssd2_inputs(case, seed))
    if kind in ("ssd2_train", "mamba3_train"):
        t = (_ssd2_inputs if kind == "ssd2_train" else _mamba3_train_inputs)(case, seed)
        for k, v in t.items():
            if k not in ("dy", "dhT"):
                v.requires_grad_(True)
        return dict(case=case, **t)
    if kind == "mamba1_scan":
        return dict(case=case, **_mamba1_scan_inputs(case, seed))
    if not kind.endswith("_decode"):
        m, x = _block(case, seed)
        return dict(case=case, block=m, x=x)
    stack, caches, token = _stack(case, seed)
    x = token.clone()
    # capture the step once, as a serving loop does; the caches go back to
    # where the conversation stood
    kept = [[t.clone() for t in vars(c).values() if torch.is_tensor(t)] for c in caches]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        stack.step_(x, caches)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        stack.step_(x, caches)
    for c, k in zip(caches, kept):
        for t, v in zip((t for t in vars(c).values() if torch.is_tensor(t)), k):
            t.copy_(v)
    return dict(case=case, stack=stack, caches=caches, token=token, x=x, graph=graph)


# ----------------------------------------------------------------------- runs --

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "ssd2":
        return mamba_hip.ssd2_fwd(s["x"], s["dt"], s["A"], s["B"], s["C"], s["D"], s["h0"], chunk_len=case["chunk"])
    if kind == "ssd2_train":
        leaves = [s[k] for k in ("x", "dt", "A", "B", "C", "D", "h0")]
        y, hT = mamba_hip.ssd2_autograd(*leaves, chunk_len=case["chunk"])
        return y, hT, torch.autograd.grad((y, hT), leaves, (s["dy"], s["dhT"]))
    if kind == "mamba3_train":
        leaves = [s[k] for k in ("v", "da", "B", "C", "gamma", "scale", "h0")]
        y, hT = mamba_hip.ssd3_autograd(*leaves, chunk_len=case["chunk"])
        return y, hT, torch.autograd.grad((y, hT), leaves, (s["dy"], s["dhT"]))
    if kind == "mamba1_scan":
        return mamba_hip.mamba1_scan(s["u"], s["delta"], s["A"], s["B"], s["C"], s["D"], s["z"])
    if kind.endswith("_decode"):
        s["x"].copy_(s["token"])
        s["graph"].replay()
        return s["x"], [_tensors(c) for c in s["caches"]]
    out, cache = s["block"].forward(s["x"])
    return out, _tensors(cache)


# ----------------------------------------------------------------------- work --

def work(case):
    """Bytes: inputs read and outputs written once (a training step reads its
    inputs once for each direction).  Operations: the SSD's chunked form at
    chunks of 64 positions, and the products around it; a backward counts
    twice its forward."""
    kind = case["kind"]
    b, l = case["b"], case.get("l", 1)
    tok = b * l
    if kind in ("ssd2", "ssd2_train"):
        h, p, g, n = (case[k] for k in "hpgn")
        e = 2 if case["dtype"] == "bf16" else 4
        io = tok * (h * p * e + h * 4 + 2 * g * n * e)
        state = b * h * p * n * 4
        flops = tok * (h * (64 * p + 4 * p * n) + g * 64 * n)
        if kind == "ssd2":
            return {"bytes": io + tok * h * p * e + state * (2 if case["h0"] else 1), "flops": flops}
        return {"bytes": 3 * io + 2 * tok * h * p * e + 4 * state, "flops": 3 * flops}
    if kind == "mamba3_train":
        h, p, n, m = (case[k] for k in ("h", "p", "n", "mimo"))
        e = 2 if case["dtype"] == "bf16" else 4
        io = tok * (m * h * (p + 2 * n) * e + 3 * h * 4)
        flops = tok * m * h * (64 * (n + p) + 4 * p * n)
        return {"bytes": 3 * io + 2 * tok * m * h * p * e + 4 * b * h * p * n * 4, "flops": 3 * flops}
    if kind == "mamba1_scan":
        d, n = case["d"], case["n"]
        return {"bytes": 4 * (4 * tok * d + 2 * tok * n + d * n + d + b * d * n), "flops": tok * d * (6 * n + 8)}
    dm, n = case["d_model"], case["n"]
    if kind == "mamba1_block":
        c = mamba_hip.Mamba1Config(dm, state_rank=n)
        mats = dm * 2 * c.d_inner + c.d_inner * (c.dt_rank + 2 * n) + c.dt_rank * c.d_inner + c.d_inner * dm
        return {"bytes": 4 * (2 * tok * dm + mats + 2 * b * c.d_inner * (n + c.conv_kernel)),
                "flops": 2 * tok * mats + tok * c.d_inner * (6 * n + 16)}
    if kind in ("mamba2_block", "mamba2_decode"):
        c = mamba_hip.Mamba2Config(dm, state_rank=n)
        h, p = c.nheads, c.per_head_dim
        mats = dm * c.d_in_proj + c.d_inner * dm
        state = 4 * b * (h * p * n + c.conv_dim * c.conv_kernel)
        if kind == "mamba2_decode":
            return {"bytes": LAYERS * (2 * mats + 2 * state) + 8 * b * dm, "flops": LAYERS * b * (2 * mats + 6 * h * p * n)}
        return {"bytes": 2 * (2 * tok * dm + mats) + state,
                "flops": 2 * tok * mats + tok * (h * (64 * p + 4 * p * n) + 64 * n)}
    c = mamba_hip.Mamba3Config(dm, state_rank=n, mimo_rank=case["mimo"])
    h, p, m = c.nheads, c.per_head_dim, c.mimo_rank
    mats = dm * c.d_in_proj + c.d_inner * dm
    state = 4 * b * (h * p * n + m * h * n + h * p + h * c.num_rope_angles)
    if kind == "mamba3_decode":
        return {"bytes": LAYERS * (2 * mats + 2 * state) + 8 * b * dm, "flops": LAYERS * b * (2 * mats + 4 * m * h * p * n)}
    e = 2 if kind == "mamba3_prefill" else 4
    return {"bytes": e * (2 * tok * dm + mats) + state,
            "flops": 2 * tok * mats + tok * m * h * (64 * (n + p) + 4 * p * n)}


# ----------------------------------------------------------------- tolerances --

def tolerance(case):
    """About four times what each path was off its 64-bit result by, as
    measured over the ranges: f32 paths 1e-6 to 4e-6, single bf16 operations
    2e-3 (the rounding of the result), bf16 blocks and stacks 3e-3 to 6e-3
    (Mamba-3's state after thousands of tokens 3e-2, from the rounded rotation
    columns, which two correct programs share)."""
    kind = case["kind"]
    if kind in ("mamba1_scan", "mamba1_block", "mamba3_block"):
        return {"rel": 1e-5}
    if case.get("dtype") == "f32":
        return {"rel": 1e-5}
    if kind in ("ssd2", "ssd2_train", "mamba3_train"):
        return {"rel": 1e-2}
    return {"rel": 2e-2}


# ------------------------------------------------------------- 64-bit results --

def _up(t):
    return t.double() if torch.is_tensor(t) else t


def _ssd64(v, da, B, C, scale, gamma, h0, steps):
    """y and final state of the SSD on fused (step, rank) rows in chunks of
    ``steps`` positions: v [b, l, m, h, p], B and C [b, l, m, h, n], the rest
    [b, l, h].  A source of an earlier step weighs scale, one of the same step
    gamma (the whole same-step block)."""
    b, l, m, h, p = v.shape
    ys, S = [], h0
    for t in range(0, l, steps):
        rows = lambda a: a[:, t:t + steps].permute(0, 3, 1, 2, 4).flatten(2, 3)  # noqa: E731  [b, h, q m, .]
        cs = da[:, t:t + steps].cumsum(1).transpose(1, 2)                         # [b, h, q]
        q = cs.shape[2]
        csf = cs.repeat_interleave(m, 2)
        sc = scale[:, t:t + steps].transpose(1, 2).repeat_interleave(m, 2)
        ga = gamma[:, t:t + steps].transpose(1, 2).repeat_interleave(m, 2)
        at = torch.arange(q, device=v.device).repeat_interleave(m)
        later, same = at[None, :] > at[:, None], at[None, :] == at[:, None]
        W = torch.exp((csf[..., :, None] - csf[..., None, :]).masked_fill(later | same, -math.inf)) * sc[..., None, :]
        W = W + same * ga[..., :, None]
        vc, Bc, Cc = rows(v), rows(B), rows(C)
        y = ((Cc @ Bc.transpose(-1, -2)) * W) @ vc + torch.exp(csf)[..., None] * (Cc @ S.transpose(-1, -2))
        S = torch.exp(cs[..., -1])[..., None, None] * S + \
            (vc * (sc * torch.exp(cs[..., -1:] - csf))[..., None]).transpose(-1, -2) @ Bc
        ys.append(y.unflatten(2, (q, m)).permute(0, 2, 3, 1, 4))
    return torch.cat(ys, 1), S


def _ssd2_64(x, dt, A, B, C, D, h0):
    b, l, h, p = x.shape
    heads = lambda t: t.repeat_interleave(h // t.shape[2], 2).unsqueeze(2)  # noqa: E731
    S = torch.zeros(b, h, p, B.shape[3], dtype=F64, device=x.device) if h0 is None else h0
    y, S = _ssd64(x.unsqueeze(2), dt * A, heads(B), heads(C), dt, dt, S, 64)
    return y.squeeze(2) + D[:, None] * x, S


def _grads64(fn, leaves, dy, dhT):
    leaves = [_up(t).detach().requires_grad_(True) for t in leaves]
    y, hT = fn(*leaves)
    return y.detach(), hT.detach(), torch.autograd.grad((y, hT), leaves, (_up(dy), _up(dhT)))


def _softplus(t):
    return torch.log1p(torch.exp(-t.abs())) + t.clamp(min=0)


def _conv64(x, window, w, bias):
    """SiLU of the causal depthwise conv over [window | x], x [b, l, c], and the new window."""
    K = w.shape[1]
    pad = torch.cat([window[:, :, 1:].transpose(1, 2), x], 1)
    y = sum(pad[:, k:k + x.shape[1]] * w[:, k] for k in range(K))
    return F.silu(y if bias is None else y + bias), pad[:, -K:].transpose(1, 2)


def _mamba1_scan64(u, delta, A, B, C, D, z, h):
    """u, delta, z [b, d, l]; B, C [b, n, l]; h [b, d, n]."""
    y = torch.empty_like(u)
    for t in range(u.shape[2]):
        dt = delta[:, :, t, None]
        h = torch.exp(dt * A) * h + dt * u[:, :, t, None] * B[:, None, :, t]
        y[:, :, t] = (h * C[:, None, :, t]).sum(2)
    return (y + D[:, None] * u) * F.silu(z), h


def _mamba1_block64(m, x):
    c = m.cfg
    b = x.shape[0]
    w = lambda t: _up(t)  # noqa: E731
    xr = _up(x) @ w(m.in_proj_w)
    u, conv = _conv64(xr[..., :c.d_inner], torch.zeros(b, c.d_inner, c.conv_kernel, dtype=F64, device=DEV),
                      w(m.conv_w), w(m.conv_b))
    dbl = u @ w(m.x_proj_w)
    r, n = c.dt_rank, c.state_rank
    dt = _softplus(dbl[..., :r] @ w(m.dt_proj_w) + w(m.dt_proj_b))
    t = lambda a: a.transpose(1, 2).contiguous()  # noqa: E731
    y, h = _mamba1_scan64(t(u), t(dt), -torch.exp(w(m.a_log)), t(dbl[..., r:r + n]), t(dbl[..., r + n:]), w(m.d),
                          t(xr[..., c.d_inner:]), torch.zeros(b, c.d_inner, n, dtype=F64, device=DEV))
    return t(y) @ w(m.out_proj_w), dict(conv=conv, ssm=h)


def _gated_norm64(y, z, gamma, eps):
    g = y * F.silu(z)
    return g * torch.rsqrt(g.square().mean(-1, keepdim=True) + eps) * gamma


def _mamba2_mixer64(m, x, conv, S, eps):
    """Mamba-2 block on x [b, l, d_model] from the cache (conv window, state)."""
    c = m.cfg
    di, gn = c.d_inner, c.ngroups * c.state_rank
    zx = x @ _up(m.in_proj_w)
    xbc, conv = _conv64(zx[..., di:di + c.conv_dim], conv, _up(m.conv_w), _up(m.conv_b))
    dt = _softplus(zx[..., di + c.conv_dim:] + _up(m.dt_bias)).clamp(*c.dt_limit)
    split = lambda t: t.unflatten(2, (c.ngroups, c.state_rank))  # noqa: E731
    y, S = _ssd2_64(xbc[..., :di].unflatten(2, (c.nheads, c.per_head_dim)), dt, -torch.exp(_up(m.a_log)),
                    split(xbc[..., di:di + gn]), split(xbc[..., di + gn:]), _up(m.d), S)
    y = _gated_norm64(y.flatten(2), zx[..., :di], _up(m.norm_w), eps)
    return y @ _up(m.out_proj_w), conv, S


def _mamba3_mixer64(m, x, S, K, V, angle):
    """Mamba-3 block on x [b, l, d_model] from the cache (state, previous rotated B, previous x, angle)."""
    c = m.cfg
    H, P, N, M, G, di, R = (c.nheads, c.per_head_dim, c.state_rank, c.mimo_rank, c.ngroups, c.d_inner, c.rope_dim)
    b, l, _ = x.shape
    proj = x @ _up(m.in_proj_w)
    z, xv, Br, Cr, dd, da, lam, rot = proj.split([di, di, M * G * N, M * G * N, H, H, H, c.num_rope_angles], -1)
    dt = _softplus(dd + _up(m.dt_bias)).clamp(*c.dt_limit)
    da = dt * -_softplus(da).clamp(min=c.a_floor)
    lam = torch.sigmoid(lam)
    gamma = lam * dt
    scale = gamma + F.pad((1 - lam[:, 1:]) * dt[:, 1:], (0, 0, 0, 1))
    th = angle[:, None] + (dt[..., None] * (c.rotation_range * math.pi * torch.tanh(rot))[:, :, None]).cumsum(1)
    k = torch.arange(R // 2, device=x.device)
    i0, i1 = (2 * k, 2 * k + 1) if M == 1 else (k, k + N // 2)
    cos, sin = torch.cos(th[:, :, None, :, :R // 2]), torch.sin(th[:, :, None, :, :R // 2])

    def rotated(raw, weight, bias):
        raw = raw.unflatten(2, (M, G, N))
        t = raw * torch.rsqrt(raw.square().mean(-1, keepdim=True) + 8.1584695e-8) * _up(weight)
        t = t.repeat_interleave(H // G, 3) + _up(bias).transpose(0, 1)
        out = t.clone()
        out[..., i0] = cos * t[..., i0] - sin * t[..., i1]
        out[..., i1] = sin * t[..., i0] + cos * t[..., i1]
        return out

    Bq, Cq = rotated(Br, m.b_norm_w, m.b_bias), rotated(Cr, m.c_norm_w, m.c_bias)
    xv = xv.unflatten(2, (H, P))
    ranks = lambda w: torch.ones(M, H, P, dtype=F64, device=x.device) if w is None else _up(w).transpose(0, 1)  # noqa: E731
    v = xv[:, :, None] * ranks(m.mimo_x)
    # the trapezoid's share of the previous token enters through the state
    seed = torch.einsum("bmhp,bmhn->bhpn", V[:, None] * ranks(m.mimo_x), K)
    S = S + (dt[:, 0] - gamma[:, 0])[..., None, None] * seed
    y, S = _ssd64(v, da, Bq, Cq, scale, gamma, S, max(1, 64 // M))
    y = y + _up(m.D)[:, None] * v
    y = (y * F.silu(z.unflatten(2, (H, P))[:, :, None] * ranks(m.mimo_z)) * ranks(m.mimo_o)).sum(2)
    return y.flatten(2) @ _up(m.out_proj_w), S, Bq[:, -1], xv[:, -1]


@torch.no_grad()
def _decode64(stack, caches, token):
    x, out = _up(token), []
    for layer, cache in zip(stack.layers, caches):
        u = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 8.1584695e-8) * _up(layer.norm_w)
        u = u[:, None]
        if isinstance(cache, mamba_hip.Mamba2Cache):
            y, conv, S = _mamba2_mixer64(layer.mixer, u, _up(cache.conv_bvk), _up(cache.ssm_bhpr), 8.1584695e-8)
            out.append(dict(conv=conv, ssm=S))
        else:
            y, S, K, V = _mamba3_mixer64(layer.mixer, u, _up(cache.ssm_bhpr), _up(cache.k_state_bmhr),
                                         _up(cache.v_state_bhp), _up(cache.angle_bha))
            out.append(dict(ssm=S, k=K, v=V))
        x = x + y[:, 0]
    return x, out


def exact(case, seed):
    kind = case["kind"]
    if kind == "ssd2":
        return _ssd2_64(*(_up(v) for v in _ssd2_inputs(case, seed).values()))
    if kind == "ssd2_train":
        t = _ssd2_inputs(case, seed)
        return _grads64(_ssd2_64, [t[k] for k in ("x", "dt", "A", "B", "C", "D", "h0")], t["dy"], t["dhT"])
    if kind == "mamba3_train":
        t = _mamba3_train_inputs(case, seed)

        def fn(v, da, B, C, gamma, scale, h0):
            return _ssd64(v, da, B, C, scale, gamma, h0, max(1, 64 // case["mimo"]))
        return _grads64(fn, [t[k] for k in ("v", "da", "B", "C", "gamma", "scale", "h0")], t["dy"], t["dhT"])
    if kind == "mamba1_scan":
        t = _mamba1_scan_inputs(case, seed)
        return _mamba1_scan64(*(_up(v) for v in t.values()),
                              torch.zeros(case["b"], case["d"], case["n"], dtype=F64, device=DEV))
    if kind.endswith("_decode"):
        return _decode64(*_stack(case, seed))
    m, x = _block(case, seed)
    c, b = m.cfg, case["b"]
    zeros = lambda *shape: torch.zeros(b, *shape, dtype=F64, device=DEV)  # noqa: E731
    with torch.no_grad():
        if kind == "mamba1_block":
            return _mamba1_block64(m, x)
        if kind == "mamba2_block":
            # the gated norm's epsilon is that of the block's type
            y, conv, S = _mamba2_mixer64(m, _up(x), zeros(c.conv_dim, c.conv_kernel),
                                         zeros(c.nheads, c.per_head_dim, c.state_rank), mamba_hip.div_eps(BF16))
            return y, dict(conv=conv, ssm=S)
        y, S, K, V = _mamba3_mixer64(m, _up(x), zeros(c.nheads, c.per_head_dim, c.state_rank),
                                     zeros(c.mimo_rank, c.nheads, c.state_rank), zeros(c.nheads, c.per_head_dim),
                                     zeros(c.nheads, c.num_rope_angles))
        return y, dict(ssm=S, k=K, v=V)
