"""Workloads of the FMM evaluator that its speed is measured on.

Every case is a call that a program using this package makes through its
public entry points: an evaluation on a tree that it holds, a time step (tree
build plus evaluation), the Barnes-Hut walk, a direct sum at chosen targets, a
batch of one generated operator, and the gradient of the order network.
Particle sets follow the distributions of fmmgen_amd/workloads.py, drawn on the
GPU.
"""
import math

import torch

from fmmgen_amd import build_tree, direct_sum
from fmmgen_amd import learned as order_net
from fmmgen_amd.operators import Library

F64 = torch.float64

# dist, n, order, theta, ncrit: the set and tree; so: source order (0 charges,
# 1 dipoles, 2 quadrupoles); pot / field: the outputs; mode: of the evaluation.
_EVAL = dict(kind="eval", so=0, pot=True, field=True, mode="plain", theta=0.5, ncrit=64)


def listed():
    return [
        # a few thousand particles: every launch counts (interactive use, a test's call)
        dict(_EVAL, name="eval_small", dist="uniform", n=2000, order=4),
        # the example's own size: 10^5 uniform charges at order 4
        dict(_EVAL, name="eval_1e5", dist="uniform", n=100_000, order=4),
        # 2^20 uniform charges at order 8 in FP64, the mid-size reference run
        dict(_EVAL, name="eval_2e20", dist="uniform", n=1 << 20, order=8),
        # clustered dipoles (a micromagnetic demagnetising field), FP32 matrix-core M2L
        dict(_EVAL, name="eval_dipole_f32", dist="plummer", n=1_000_000, order=6, theta=0.4, ncrit=32, so=1,
             pot=False, mode="f32"),
        # the method without the network at 1e-6 on clustered charges, FP64
        dict(_EVAL, name="eval_blobs_plain", dist="blobs", n=1 << 22, order=10),
        # the headline: learned orders and opening angle at 1e-6, FP32
        dict(_EVAL, name="eval_blobs_learned", dist="blobs", n=1 << 22, order=12, mode="learned"),
        # the largest: 2^24 half uniform, half Plummer, learned orders with the BF16x3 M2L
        dict(_EVAL, name="eval_mixed_learned_bf16x3", dist="mixed", n=1 << 24, order=12, ncrit=128,
             mode="learned_bf16x3"),
        # one step of a particle simulation: the particles have moved, so tree, lists and field are new
        dict(_EVAL, name="step_blobs", kind="step", dist="blobs", n=300_007, order=6),
        # Barnes-Hut on the mid-size set
        dict(_EVAL, name="bh_2e20", kind="bh", dist="uniform", n=1 << 20, order=8),
        # a check of a field at 4096 sampled targets by the FP64 direct sum
        dict(kind="direct", name="direct_4096", dist="uniform", n=1 << 20, targets=4096, so=0, pot=True, field=True),
        # the generated operators called in a batch by a program with a tree of its own
        dict(kind="op", name="op_m2l_batch", op="M2L", order=10, batch=20_000, so=0, pot=True, field=True),
        # one gradient of the order network at the training's batch
        dict(kind="train", name="train_grad", batch=2048),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _flavour(rng):
    """(source order, potential, field) of a compiled variant, charges with both outputs mostly."""
    return rng.choice([(0, True, True)] * 5 + [(0, True, False), (0, False, True), (1, False, True), (1, False, True),
                                               (2, True, True)])


def draw(rng):
    kind = rng.choice(["eval"] * 7 + ["step"] * 2 + ["bh", "direct", "op", "train"])
    if kind == "train":
        return dict(kind="train", batch=_log_uniform(rng, 256, 8192))
    so, pot, field = _flavour(rng)
    if kind == "op":
        op = rng.choice(["P2M", "M2M", "M2L", "M2L", "L2L", "L2P", "M2P"])
        lo, hi = so + (1 if field else 0), 12 if so == 0 else 8
        if op == "P2M" and so:
            op = "M2M"
        return dict(kind="op", op=op, order=rng.randint(max(lo, 1), hi), batch=_log_uniform(rng, 64, 20_000), so=so,
                    pot=pot, field=field)
    dist = rng.choice(["uniform", "blobs", "plummer", "mixed"])
    if kind == "direct":
        return dict(kind="direct", dist=dist, n=_log_uniform(rng, 1000, 1 << 20), targets=_log_uniform(rng, 100, 4096),
                    so=so, pot=pot, field=field)
    mode = "plain" if kind == "bh" else rng.choice(["plain", "plain", "plain", "f32", "bf16x3", "learned",
                                                    "learned_bf16x3"])
    if kind == "step" and mode.startswith("learned"):
        mode = "f32"
    if mode.startswith("learned"):
        so, pot, field = 0, True, True
        n, order, theta = _log_uniform(rng, 1 << 16, 1 << 22), 12, 0.5
    else:
        order = rng.randint(max(2, so + 1), 10 if so == 0 else 8)
        theta = rng.choice([0.4, 0.5, 0.5, 0.55])
        top = {"eval": 1 << 21, "step": 1 << 20, "bh": 1 << 20}[kind]
        n = _log_uniform(rng, 1000, top if so == 0 and theta >= 0.5 else top // 4)
        if kind == "bh":
            order = min(order, 8)
    return dict(kind=kind, dist=dist, n=n, order=order, theta=theta, ncrit=rng.choice([32, 64, 64, 128]), so=so,
                pot=pot, field=field, mode=mode)


# ------------------------------------------------------------------ inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _uniform(shape, g):
    return torch.rand(*shape, generator=g, device="cuda", dtype=F64)


def _normal(shape, g):
    return torch.randn(*shape, generator=g, device="cuda", dtype=F64)


def _plummer(n, g, a, rmax=1.0):
    """Plummer sphere truncated at rmax: r = a / sqrt(X^(-2/3) - 1)."""
    x = _uniform((n,), g) * (1.0 + (a / rmax) ** 2) ** -1.5
    r = a / torch.sqrt(x.clamp_min(1e-12) ** (-2.0 / 3.0) - 1.0)
    v = _normal((n, 3), g)
    return v / v.norm(dim=1, keepdim=True) * r[:, None]


def _positions(dist, n, g):
    if dist == "uniform":
        return _uniform((n, 3), g)
    if dist == "plummer":
        return _plummer(n, g, 0.1)
    if dist == "mixed":
        h = n // 2
        p = torch.cat([_uniform((h, 3), g), _plummer(n - h, g, 0.05) + 0.5])
    else:  # 16 Gaussian blobs and 20% uniform background
        nbg = int(round(0.2 * n))
        centres, sigma = _uniform((16, 3), g), 0.01 + 0.09 * _uniform((16,), g)
        which = torch.randint(0, 16, (n - nbg,), generator=g, device="cuda")
        p = torch.cat([centres[which] + _normal((n - nbg, 3), g) * sigma[which, None], _uniform((nbg, 3), g)])
    return p[torch.randperm(n, generator=g, device="cuda")].contiguous()


def _sources(so, n, g):
    if so == 0:
        return 2.0 * _uniform((n, 1), g) - 1.0
    v = _normal((n, 3 if so == 1 else 6), g)
    return v / v.norm(dim=1, keepdim=True) * torch.exp(0.5 * _normal((n, 1), g))


def _outsz(c):
    return (1 if c["pot"] else 0) + (3 if c["field"] else 0)


def _nterms(p):
    return (p + 1) * (p + 2) * (p + 3) // 6 if p >= 0 else 0


def _sizes(op, c):
    """(inputs, outputs) of one operator application."""
    so, p = c["so"], c["order"]
    ms, ls = _nterms(p) - _nterms(so - 1), _nterms(p - so)
    return {"P2M": (1, ms), "M2M": (ms, ms), "M2L": (ms, ls), "L2L": (ls, ls), "L2P": (ls, _outsz(c)),
            "M2P": (ms, _outsz(c))}[op]


def _op_inputs(c, seed):
    g = _generator(seed)
    b, (nin, nout) = c["batch"], _sizes(c["op"], c)
    far = 2.0 if c["op"] in ("M2L", "M2P") else 0.0  # well separated, or inside a cell of half-width 1
    d = 2.0 * _uniform((b, 3), g) - 1.0
    d = d + far * torch.sign(d)
    return d, _normal((b, nin), g), torch.zeros(b, nout, dtype=F64, device="cuda")


def _train_inputs(c, seed):
    g, b = _generator(seed), c["batch"]
    X = torch.randn(b, order_net.F, generator=g, device="cuda")
    T = -4.0 + 2.0 * torch.randn(b, order_net.O, generator=g, device="cuda")
    mask = (torch.rand(b, order_net.O, generator=g, device="cuda") < 0.95).float()
    return X, T, mask, order_net.init_params(seed % (1 << 31))


def _set(c, seed):
    g = _generator(seed)
    return _positions(c["dist"], c["n"], g).contiguous(), _sources(c["so"], c["n"], g).contiguous()


def _targets(c, seed):
    return torch.randperm(c["n"], generator=_generator(seed + 1), device="cuda")[:min(c["targets"], c["n"])].contiguous()


def _tree(c, pos, S):
    return build_tree(pos, S, c["n"], c["ncrit"], c["order"], c["theta"], source_order=c["so"], potential=c["pot"],
                      field=c["field"])


def prepare(case, seed):
    c = case
    if c["kind"] == "op":
        d, a, out = _op_inputs(c, seed)
        x, y, z = (d[:, k].contiguous() for k in range(3))
        return dict(case=c, lib=Library(c["so"], c["pot"], c["field"]), xyz=(x, y, z), a=a, out=out)
    if c["kind"] == "train":
        X, T, mask, params = _train_inputs(c, seed)
        return dict(case=c, X=X, T=T, mask=mask, params=params)
    pos, S = _set(c, seed)
    if c["kind"] == "direct":
        return dict(case=c, pos=pos, S=S, targets=_targets(c, seed))
    F = torch.empty(c["n"], _outsz(c), dtype=F64, device="cuda")
    s = dict(case=c, pos=pos, S=S, F=F)
    if c["kind"] != "step":
        s["tree"] = t = _tree(c, pos, S)
        if c["mode"].startswith("learned"):
            params, margin, _ = order_net.load()
            t.set_model(params, 1e-6, margin, thetas=[0.5, 0.55])
    return s


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "eval":
        return s["tree"].compute_field_fmm(s["F"], mode=c["mode"])
    if c["kind"] == "step":
        return _tree(c, s["pos"], s["S"]).compute_field_fmm(s["F"], mode=c["mode"])
    if c["kind"] == "bh":
        return s["tree"].compute_field_bh(s["F"])
    if c["kind"] == "direct":
        return direct_sum(s["pos"], s["S"], s["targets"], source_order=c["so"], outsz=_outsz(c))
    if c["kind"] == "op":
        s["out"].zero_()
        getattr(s["lib"], c["op"])(*s["xyz"], s["a"], s["out"], c["order"])
        return s["out"]
    loss, g = order_net.grad(s["X"], s["T"], s["mask"], s["params"])
    return {"loss": loss, "grad": g}


# ------------------------------------------------------------------ work

def _pair_flops(so):
    return {0: 20, 1: 60, 2: 130}[so]


def _m2l_macs(p, so):
    """Multiply-adds of one M2L pair over independent rows and columns (harmonic functions: 2n + 1 of degree n)."""
    return sum((2 * n + 1) * sum(2 * m + 1 for m in range(so, p - n + 1)) for n in range(p - so + 1))


def work(case):
    """Bytes and operations of one pass.  The pairs of a tree are estimates:
    about 4700 near-field pairs and 27 translations a particle at 64 particles
    a leaf and an opening angle of 0.5 (blobs of 2^22), scaled by theta^-3."""
    c = case
    if c["kind"] == "train":
        h, f, o = order_net.H, order_net.F, order_net.O
        n = f * h + h * h + h * o
        return {"bytes": 4 * c["batch"] * (f + 2 * o) + 8 * (n + 2 * h + o), "flops": 6 * c["batch"] * n}
    if c["kind"] == "op":
        nin, nout = _sizes(c["op"], c)
        macs = {"M2L": _m2l_macs(c["order"], c["so"])}.get(c["op"], 4 * max(nin, nout))
        return {"bytes": 8 * c["batch"] * (3 + nin + nout), "flops": 2 * c["batch"] * macs}
    n, ss = c["n"], {0: 1, 1: 3, 2: 6}[c["so"]]
    if c["kind"] == "direct":
        t = min(c["targets"], n)
        return {"bytes": 8 * n * (3 + ss) + 8 * t * (1 + _outsz(c)), "flops": _pair_flops(c["so"]) * n * t}
    scale = (0.5 / c["theta"]) ** 3
    near = min(4700.0 * c["ncrit"] / 64 * scale, n)
    far = 27.0 * 64 / c["ncrit"] * scale if n > 8 * c["ncrit"] else 0.0
    order = c["order"] - 4 if c["mode"].startswith("learned") else c["order"]  # about 8 on average at 1e-6
    return {"bytes": 8 * n * (3 + ss + _outsz(c)),
            "flops": n * (near * _pair_flops(c["so"]) + far * 2 * _m2l_macs(order, c["so"]))}


# ------------------------------------------------------------------ exact values

def _monomials(lo, hi):
    """Multi-indices of degree lo .. hi in the expansions' order."""
    return [(d - a, a - b, b) for d in range(lo, hi + 1) for a in range(d + 1) for b in range(a + 1)]


def _derivatives(x, y, z, p):
    """{n: d^n (1/R)} for |n| <= p, by |n| R^2 D_n = -(2|n| - 1) sum x_i n_i D_{n-e_i} - (|n| - 1) sum n_i (n_i - 1) D_{n-2e_i}."""
    r2, v = x * x + y * y + z * z, (x, y, z)
    D = {(0, 0, 0): r2.rsqrt()}
    for n in _monomials(1, p):
        d, acc = sum(n), 0.0
        for i in range(3):
            for k, w in ((1, -(2 * d - 1) * n[i]), (2, -(d - 1) * n[i] * (n[i] - 1))):
                if w:
                    m = tuple(n[j] - (k if j == i else 0) for j in range(3))
                    acc = acc + (w / d) * D[m] * (v[i] if k == 1 else 1.0)
        D[n] = acc / r2
    return D


def _shift(n, axis):
    return tuple(n[j] + (1 if j == axis else 0) for j in range(3))


def _outputs(D, moments, c):
    """Potential sum M_n D_n and field -grad, stacked on the last axis."""
    out = [sum(w * D[n] for n, w in moments)] if c["pot"] else []
    if c["field"]:
        out += [-sum(w * D[_shift(n, a)] for n, w in moments) for a in range(3)]
    return torch.stack(out, -1)


def _direct_exact(pos, S, targets, c):
    n, so = pos.shape[0], c["so"]
    out = torch.empty(targets.shape[0], _outsz(c), dtype=F64, device="cuda")
    rows = max(1, (1 << 25) // n)
    idx = _monomials(so, so)
    for b in range(0, targets.shape[0], rows):
        t = targets[b:b + rows]
        dx, dy, dz = (pos[t, k][:, None] - pos[None, :, k] for k in range(3))
        me = torch.arange(t.shape[0], device="cuda")
        dx[me, t] = 1.0  # the target itself: no source
        w = [S[None, :, k].expand(t.shape[0], n).clone() for k in range(S.shape[1])]
        for v in w:
            v[me, t] = 0.0
        if so == 0:
            r = (dx * dx + dy * dy + dz * dz).rsqrt()
            q = w[0] * r
            q3 = q * r * r
            cols = [q.sum(1)] if c["pot"] else []
            cols += [(q3 * v).sum(1) for v in (dx, dy, dz)] if c["field"] else []
            out[b:b + rows] = torch.stack(cols, 1)
        else:
            D = _derivatives(dx, dy, dz, so + (1 if c["field"] else 0))
            out[b:b + rows] = _outputs(D, list(zip(idx, w)), c).sum(1)
    return out


def _power(x, n):
    v = 1.0
    for k in range(3):
        v = v * x[k] ** n[k] / math.factorial(n[k])
    return v


def _op_exact(c, seed):
    d, a, _ = _op_inputs(c, seed)
    op, p, so = c["op"], c["order"], c["so"]
    x = (d[:, 0], d[:, 1], d[:, 2])
    M, L = _monomials(so, p), _monomials(0, p - so)
    ms, ls = {n: i for i, n in enumerate(M)}, {n: i for i, n in enumerate(L)}

    def minus(n, k):
        return tuple(n[j] - k[j] for j in range(3))

    def plus(n, k):
        return tuple(n[j] + k[j] for j in range(3))
    if op == "P2M":
        return torch.stack([a[:, 0] * (-1) ** sum(n) * _power(x, n) for n in M], 1)
    if op == "M2P":
        return _outputs(_derivatives(*x, p + 1), [(n, a[:, i]) for n, i in ms.items()], c)
    if op == "L2P":
        def at(axis):
            t = torch.zeros_like(x[0])
            for n, i in ls.items():
                m = n if axis is None else minus(n, _shift((0, 0, 0), axis))
                if min(m) >= 0:
                    t = t + a[:, i] * _power(x, m)
            return t
        out = [at(None)] if c["pot"] else []
        return torch.stack(out + ([-at(k) for k in range(3)] if c["field"] else []), 1)
    pw = {n: _power(x, n) for n in _monomials(0, p)} if op in ("M2M", "L2L") else None
    cols = []
    if op == "M2L":
        D = _derivatives(*x, p)
        for n in L:
            cols.append(sum(D[plus(n, m)] * a[:, i] for m, i in ms.items() if sum(n) + sum(m) <= p))
    elif op == "M2M":
        for n in M:
            cols.append(sum(a[:, i] * pw[minus(n, m)] for m, i in ms.items() if min(minus(n, m)) >= 0))
    else:
        for n in L:
            cols.append(sum(a[:, i] * pw[minus(m, n)] for m, i in ls.items() if min(minus(m, n)) >= 0))
    return torch.stack([v + torch.zeros_like(x[0]) for v in cols], 1)


def _train_exact(c, seed):
    X, T, mask, params = (v.double() for v in _train_inputs(c, seed))
    p = params.requires_grad_(True)
    f, h, o = order_net.F, order_net.H, order_net.O
    v, at = X, 0
    for nin, nout, last in ((f, h, False), (h, h, False), (h, o, True)):
        W, b = p[at:at + nin * nout].view(nout, nin), p[at + nin * nout:at + nin * nout + nout]
        at += nin * nout + nout
        v = v @ W.t() + b
        v = v if last else torch.relu(v)
    loss = (((v - T) * mask) ** 2).sum() / mask.sum()
    loss.backward()
    return {"loss": loss.detach().reshape(1), "grad": p.grad}


def exact(case, seed):
    """The direct sum for particle sets up to 2^17 (and for sampled targets of any set), the operators' series, the
    network's gradient; None for larger sets."""
    c = case
    if c["kind"] == "train":
        return _train_exact(c, seed)
    if c["kind"] == "op":
        return _op_exact(c, seed)
    if c["kind"] == "direct":
        return _direct_exact(*_set(c, seed), _targets(c, seed), c)
    if c["n"] > (1 << 17) or (c["so"] and c["n"] > (1 << 16)):
        return None
    return _direct_exact(*_set(c, seed), torch.arange(c["n"], device="cuda"), c)
