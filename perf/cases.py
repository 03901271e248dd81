"""The measured workloads of the shift-window operators.

Twelve listed cases, and ``draw`` for more of the same ranges.  A case names an
operator (``op``), a shift table (``table`` and radius ``R``), the image shape
and the options a caller passes; ``train`` cases run the forward and the
autograd backward with given upstream gradients, the others run the forward
under ``no_grad`` as inference does.  Shapes are those of ``bench.py``, of
``neural_shift_cuda_amd/workloads.py`` and of the tests, or plain image sizes.
"""
from __future__ import annotations

import math

import torch

import neural_shift_cuda as nsc
from neural_shift_cuda.metropolis import metropolis_aggregate
from neural_shift_cuda_amd.ops import normalized_accumulate_uz_mixed
from neural_shift_cuda_amd.workloads import halfplane_rows

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32,
          "fp64": torch.float64}
BYTES = {"fp16": 2, "bf16": 2, "fp32": 4, "fp64": 8}
EPS = 1e-6  # metropolis_aggregate's default


def listed():
    return [
        # Neighbour features of a training patch batch (the 64 x 64 patches a
        # denoiser trains on): a small call, where launches and host time count.
        _case("gather_patches_bf16", op="shift_gather", table="half", R=5, B=8, C=3, H=64, W=64,
              dtype="bf16", train=True),
        # (centre, neighbour) pairs for a similarity network, both directions.
        _case("pair_gather_bf16", op="pair_gather", table="half", R=5, B=8, C=3, H=256, W=256,
              dtype="bf16", train=True),
        # One small image, inference: the smallest accumulation a caller makes.
        _case("accumulate_small", op="accumulate", table="half", R=3, B=1, C=1, H=256, W=256,
              dtype="fp32", train=False, weights="boxed"),
        # Mixed-precision training batch of grey images.
        _case("accumulate_fp16_train", op="accumulate", table="half", R=7, B=4, C=1, H=512, W=512,
              dtype="fp16", train=True, weights="boxed"),
        # Full photographs as they come: no side a multiple of anything, colour,
        # the box mask left to the op.
        _case("accumulate_photo_train", op="accumulate", table="half", R=5, B=2, C=3, H=321, W=481,
              dtype="fp32", train=True, box_forward=True),
        # The largest: one 8192 x 8192 image, 22.8 GB of weights.
        _case("accumulate_8k_train", op="accumulate", table="half", R=6, B=1, C=1, H=8192, W=8192,
              dtype="fp32", train=True, weights="boxed"),
        # Row-stochastic denoising over the full window, called as documented
        # (the weight check included).
        _case("normalized_window_train", op="normalized", table="window", R=5, B=16, C=3, H=256,
              W=256, dtype="fp32", train=True, validate=True),
        # Attention logits in half precision with outliers, as the attention
        # layers call it: D and log C, box mask in the op, no weight check.
        _case("normalized_logits_fp16_train", op="normalized", table="half", R=7, B=4, C=1, H=512,
              W=512, dtype="fp16", train=True, log=True, box_forward=True, degree=True),
        # A wide search window on one large image, inference.
        _case("normalized_wide", op="normalized", table="half", R=10, B=1, C=1, H=1024, W=1024,
              dtype="fp32", train=False, box_forward=True, degree=True),
        # A one-head attention layer: one weight plane for the three channels,
        # an image size that no tile divides.
        _case("normalized_one_head_train", op="normalized", table="half", R=5, B=8, C=3, H=250,
              W=250, dtype="fp32", train=True, box_forward=True, shared=True, degree=True),
        # One weight per transform (group-averaged denoising), full window.
        _case("scalar_window_train", op="scalar", table="window", R=5, B=16, C=3, H=256, W=256,
              dtype="fp32", train=True),
        # Metropolis-Hastings aggregation in training, a large image.
        _case("metropolis_train", op="metropolis", table="half", R=6, B=1, C=1, H=2048, W=2048,
              dtype="fp32", train=True, use_box=True),
    ]


def _case(name=None, *, op, table, R, B, C, H, W, dtype, train, weights="plain", log=False,
          validate=False, box_forward=False, periodic=False, shared=False, degree=False, heads=0,
          use_box=False):
    case = {"op": op, "table": table, "R": R, "B": B, "C": C, "H": H, "W": W, "dtype": dtype,
            "train": train}
    if op in ("accumulate", "normalized"):
        case.update(weights=weights, log=log, validate=validate, box_forward=box_forward,
                    periodic=periodic, shared=shared, degree=degree, heads=heads)
    if op == "metropolis":
        case["use_box"] = use_box
    return case if name is None else {"name": name, **case}


# Most weight elements (S * B * C * H * W) of a drawn case; the largest listed
# case has 5.7e9.
_DRAWN_ELEMENTS = 8e8


def _side(rng, most):
    """A side from 48 to `most`, even over its logarithm; half of them as drawn
    (mostly no multiple of anything), half rounded to a multiple of 16."""
    n = int(round(math.exp(rng.uniform(math.log(48), math.log(most)))))
    return n if rng.random() < 0.5 else max(48, n // 16 * 16)


def draw(rng):
    """One more case: any operator, sizes over the whole range."""
    op = rng.choice(["shift_gather", "pair_gather", "accumulate", "accumulate", "accumulate",
                     "normalized", "normalized", "normalized", "mixed", "scalar", "metropolis"])
    train = rng.random() < 0.6
    table = rng.choice(["half", "half", "window"])
    R = rng.choice([3, 4, 5, 5, 6, 7, 8, 10]) if table == "half" else rng.choice([2, 3, 4, 5, 5, 7])
    B, C = rng.choice([1, 2, 4, 8, 16]), rng.choice([1, 1, 3])
    opts = {}
    if op in ("shift_gather", "pair_gather"):
        dtype = rng.choice(["bf16", "fp16", "fp32"])
        R, C = min(R, 7), rng.choice([1, 3, 8])
    elif op == "accumulate":
        dtype = rng.choice(["fp32", "fp32", "fp16", "bf16", "fp64"])
        mode = rng.choice(["boxed", "box_forward", "periodic"])
        opts = {"weights": "boxed" if mode == "boxed" else "plain",
                "box_forward": mode == "box_forward", "periodic": mode == "periodic",
                "shared": rng.random() < 0.25}
    elif op == "normalized":
        dtype = rng.choice(["fp32", "fp32", "fp16", "bf16", "fp64"])
        mode = rng.choice(["plain", "box_forward", "box_forward", "periodic"])
        opts = {"log": rng.random() < 0.4, "validate": rng.random() < 0.4,
                "box_forward": mode == "box_forward", "periodic": mode == "periodic",
                "shared": rng.random() < 0.25, "degree": rng.random() < 0.5}
    elif op == "mixed":  # several heads, mixed to the channels
        op, dtype, train = "normalized", rng.choice(["fp32", "fp16"]), False
        C = 3
        opts = {"heads": rng.choice([2, 4]), "box_forward": rng.random() < 0.7, "degree": True}
    elif op == "scalar":
        dtype = rng.choice(["fp32", "fp32", "fp16", "fp64"])
    else:
        dtype, table = rng.choice(["fp32", "fp32", "fp16"]), "half"
        opts = {"use_box": rng.random() < 0.7}
    H = _side(rng, 2048)
    W = H if rng.random() < 0.4 else _side(rng, 2048)
    S = len(_rows({"table": table, "R": R}))
    while S * B * C * H * W > _DRAWN_ELEMENTS:
        if B > 1:
            B //= 2
        else:
            H, W = max(48, int(H * 0.7)), max(48, int(W * 0.7))
    return _case(op=op, table=table, R=R, B=B, C=C, H=H, W=W, dtype=dtype, train=train, **opts)


def _rows(case):
    R = case["R"]
    if case["table"] == "half":
        return halfplane_rows(R)
    return [(dx, dy, 0) for dx in range(-R, R + 1) for dy in range(-R, R + 1)]


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _image(shape, g):
    """Piecewise-smooth images in about [0, 1] with noise of sd 25/255."""
    B, C, H, W = shape
    img = torch.zeros(shape, device=DEV)
    hh = torch.arange(H, device=DEV, dtype=torch.float32)[:, None] / H
    ww = torch.arange(W, device=DEV, dtype=torch.float32)[None, :] / W
    corner = torch.rand(8, 4, B, C, 1, 1, generator=g, device=DEV)
    level = torch.rand(9, 3, B, C, 1, 1, generator=g, device=DEV)
    for k in range(8):
        h0, h1, w0, w1 = corner[k]
        inside = ((hh >= torch.minimum(h0, h1)) & (hh < torch.maximum(h0, h1))
                  & (ww >= torch.minimum(w0, w1)) & (ww < torch.maximum(w0, w1)))
        img = torch.where(inside, level[k, 0], img)
    fh, fw, phi = level[8]
    img += 0.1 * torch.sin(2 * math.pi * ((1 + 7 * fh) * hh + (1 + 7 * fw) * ww + phi))
    img += (25.0 / 255.0) * torch.randn(shape, generator=g, device=DEV)
    return img


def _normal(shape, g):
    return torch.randn(shape, generator=g, device=DEV)


def _planes(case, g, rows):
    """The (S*B, planes, H, W) weights or logits, made shift by shift."""
    B, H, W = case["B"], case["H"], case["W"]
    n = case.get("heads") or (1 if case.get("shared") else case["C"])
    out = torch.empty((len(rows) * B, n, H, W), dtype=DTYPES[case["dtype"]], device=DEV)
    for s, (dx, dy, _) in enumerate(rows):
        z = _normal((B, n, H, W), g)
        if case.get("log"):
            z *= 2.0
            u = torch.rand((B, n, H, W), generator=g, device=DEV)
            z = torch.where(u < 0.005, -80.0, torch.where(u > 0.995, 80.0, z))
        else:
            z = torch.nn.functional.softplus(z)
        if case.get("weights") == "boxed":
            z *= _box(H, W, dx, dy, z.dtype)
        out[s * B:(s + 1) * B] = z
    return out


def _inputs(case, seed):
    """The tensors of a case, without gradient state."""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    B, C, H, W = shape = case["B"], case["C"], case["H"], case["W"]
    op, dt = case["op"], DTYPES[case["dtype"]]
    acc = torch.float64 if dt == torch.float64 else torch.float32
    rows = _rows(case)
    S = len(rows)
    t = {"x": _image(shape, g).to(dt)}
    if op in ("accumulate", "normalized"):
        t["w"] = _planes(case, g, rows)
        if case["heads"]:
            t["mix"] = torch.softmax(_normal((C, case["heads"]), g), 1).to(dt)
    elif op == "scalar":
        t["w"] = torch.softmax(_normal((S, B, C), g), 0).to(dt)
    elif op == "metropolis":
        t["w"] = _planes(case, g, rows).view(S, B, C, H, W).transpose(0, 1).contiguous()
    if case["train"]:
        if op in ("shift_gather", "pair_gather"):
            k = C if op == "shift_gather" else 2 * C
            t["g0"] = torch.empty((S * B, k, H, W), dtype=dt, device=DEV)
            for s in range(S):
                t["g0"][s * B:(s + 1) * B] = _normal((B, k, H, W), g)
        else:
            out = dt if op == "metropolis" else acc
            t["g0"] = _normal(shape, g).to(out)
            t["g1"] = _normal(shape, g).to(out)
    return t, rows


def prepare(case, seed):
    t, rows = _inputs(case, seed)
    state = {"case": case, **t}
    if case["op"] == "metropolis":
        state["shifts"] = [(dx, dy, bool(inv)) for dx, dy, inv in rows]
    else:
        cols = 2 if case["op"] in ("shift_gather", "pair_gather", "scalar") else 3
        state["shifts"] = torch.tensor([r[:cols] for r in rows], dtype=torch.int64, device=DEV)
    if case["train"]:
        state["x"].requires_grad_(True)
        if "w" in state:
            state["w"].requires_grad_(True)
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _forward(state):
    """The outputs of a case's op, by name, the differentiable ones first."""
    case, x, shifts = state["case"], state["x"], state["shifts"]
    op = case["op"]
    if op in ("shift_gather", "pair_gather"):
        fn = nsc.shift_gather if op == "shift_gather" else nsc.pair_gather
        out, mask = fn(x, shifts)
        return {"out": out, "mask": mask}
    if op == "scalar":
        U, Z = nsc.accumulate_uz_scalar(x, state["w"], shifts)
        return {"U": U, "Z": Z}
    if op == "metropolis":
        Wx, d_hat = metropolis_aggregate(state["w"], x, shifts, case["use_box"])
        return {"Wx": Wx, "d_hat": d_hat}
    flags = {"periodic_inverse": case["periodic"], "box_forward": case["box_forward"]}
    if case["heads"]:
        D, log_C = normalized_accumulate_uz_mixed(x, state["w"], state["mix"], shifts,
                                                  return_log_degree=True, **flags)
        return {"D": D, "log_C": log_C}
    flags["shared_weights"] = case["shared"]
    if op == "accumulate":
        U, Z = nsc.accumulate_uz(x, state["w"], shifts, **flags)
        return {"U": U, "Z": Z}
    out = nsc.normalized_accumulate_uz(x, state["w"], shifts, log_weights=case["log"],
                                       return_log_degree=case["degree"],
                                       validate=case["validate"], **flags)
    return {"D": out[0], "log_C": out[1]} if case["degree"] else {"D": out}


def run(state):
    if not state["case"]["train"]:
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    names = [k for k in out if out[k].requires_grad and k != "mask"]
    leaves = {"grad_x": state["x"]}
    if "w" in state:
        leaves["grad_w"] = state["w"]
    upstream = [state["g0"], state.get("g1")][:len(names)]
    grads = torch.autograd.grad([out[k] for k in names], list(leaves.values()), upstream)
    return {**{k: v.detach() for k, v in out.items()}, **dict(zip(leaves, grads))}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    """Each call of a pass (forward, backward) reads each of its inputs once
    and writes each of its outputs once; the weights are read by both calls."""
    e = BYTES[case["dtype"]]
    a = 8 if case["dtype"] == "fp64" else 4
    rows = _rows(case)
    S, B, C = len(rows), case["B"], case["C"]
    P = case["H"] * case["W"]
    N = B * C * P
    terms = sum(2 if r[2] else 1 for r in rows)
    op, train = case["op"], case["train"]
    if op in ("shift_gather", "pair_gather"):
        stack = e * S * N * (2 if op == "pair_gather" else 1)
        n = e * N + stack + e * S * B * P
        if train:
            n += stack + e * N
        return {"bytes": n, "flops": S * N if train else 0}
    if op == "scalar":
        n = e * N + 2 * a * N + e * S * B * C
        if train:
            n += e * N + 2 * a * N + e * N + 2 * e * S * B * C
        return {"bytes": n, "flops": S * N * (2 + (4 if train else 0))}
    planes = case.get("heads") or (1 if case.get("shared") else C)
    Wt = S * B * planes * P
    if op == "metropolis":
        n = e * (Wt + N) + 2 * e * N
        if train:
            n += e * (Wt + N) + a * N + 3 * e * N + e * (Wt + N)
        return {"bytes": n, "flops": terms * N * (6 + (10 if train else 0))}
    n = e * (Wt + N) + 2 * a * N
    if train:
        n += e * (Wt + N) + (4 if op == "normalized" else 2) * a * N + e * (Wt + N)
    per = 5 if op == "normalized" else 3
    return {"bytes": n, "flops": terms * N * (per + (2 * per if train else 0))}


# ---------------------------------------------------------------------------
# Tolerances and the exact results
# ---------------------------------------------------------------------------

def tolerance(case):
    """About four times what the outputs are from ``exact`` over the listed
    cases and two dozen drawn ones."""
    dt, op, train = case["dtype"], case["op"], case["train"]
    if op in ("shift_gather", "pair_gather") and not train:
        return "exact"  # copies
    if op == "metropolis" and train:
        # grad_w routes a degree gradient by the order of two degrees, which
        # their rounding decides where they are nearly equal (the fused
        # backward against the explicit-edge path: 2.4e-4, largest 4e-2)
        return {"rel": 1e-3 if dt == "fp32" else 4e-3, "max": 0.2}
    if dt in ("fp16", "bf16") and (train or op == "metropolis"):
        # the rounding of 16-bit outputs: 2.1e-4, 1.7e-3
        return {"rel": 1e-3, "max": 2e-3} if dt == "fp16" else {"rel": 7e-3, "max": 1.6e-2}
    if case.get("heads") and dt == "fp16":
        return {"rel": 4e-5, "max": 4e-4}  # mixed weights may be rounded to 16 bits
    if dt == "fp64":
        return {"rel": 1e-14, "max": 1e-12}
    if op == "normalized":
        return {"rel": 5e-6, "max": 2e-4}
    return {"rel": 2e-6, "max": 2e-5}


def _box(H, W, dx, dy, dtype=torch.float64):
    h = torch.arange(H, device=DEV) + dx
    w = torch.arange(W, device=DEV) + dy
    return (((h >= 0) & (h < H))[:, None] & ((w >= 0) & (w < W))[None, :]).to(dtype)


def _at(t, dx, dy):
    """t at p + s."""
    return torch.roll(t, (-dx, -dy), (-2, -1))


def _back(t, dx, dy):
    """t at p - s: the adjoint of `_at`."""
    return torch.roll(t, (dx, dy), (-2, -1))


def exact(case, seed):
    t, rows = _inputs(case, seed)
    op = case["op"]
    x = t["x"].double()
    if op in ("shift_gather", "pair_gather"):
        return _exact_gather(case, t, x, rows)
    if op == "scalar":
        return _exact_scalar(case, t, x, rows)
    if op == "metropolis":
        return _exact_metropolis(case, t, x, rows)
    return _exact_accumulate(case, t, x, rows)


def _exact_gather(case, t, x, rows):
    H, W, B, C = case["H"], case["W"], case["B"], case["C"]
    pair = case["op"] == "pair_gather"
    out, mask, gx = [], [], torch.zeros_like(x)
    for s, (dx, dy, _) in enumerate(rows):
        v = _at(x, dx, dy)
        out.append(torch.cat([x, v], 1) if pair else v)
        mask.append(_box(H, W, dx, dy).expand(B, 1, H, W))
        if case["train"]:
            g = t["g0"][s * B:(s + 1) * B].double()
            gx += _back(g[:, -C:], dx, dy)
            if pair:
                gx += g[:, :C]
    got = {"out": torch.cat(out), "mask": torch.cat(mask)}
    return {**got, "grad_x": gx} if case["train"] else got


def _exact_scalar(case, t, x, rows):
    U, Z, gx = torch.zeros_like(x), torch.zeros_like(x), torch.zeros_like(x)
    gw = []
    for s, (dx, dy, _) in enumerate(rows):
        ws = t["w"][s].double()[..., None, None]
        v = _at(x, dx, dy)
        U += ws * v
        Z += ws
        if case["train"]:
            gU, gZ = t["g0"].double(), t["g1"].double()
            gw.append((gU * v + gZ).sum((-2, -1)))
            gx += _back(ws * gU, dx, dy)
    got = {"U": U, "Z": Z}
    return {**got, "grad_x": gx, "grad_w": torch.stack(gw)} if case["train"] else got


def _exact_accumulate(case, t, x, rows):
    """accumulate and normalized: a normalized result is U / Z of the weights
    (their exponentials for logits), and its gradients are the accumulation's
    with gU = gD / Z and gZ = (gL - gD D) / Z."""
    H, W, B = case["H"], case["W"], case["B"]

    def plane(s, dx, dy):
        """Weights of one shift, the forward box, the mirror's box."""
        ws = t["w"][s * B:(s + 1) * B].double()
        if case["log"]:
            ws = ws.exp()
        if case["heads"]:
            ws = (t["mix"].double()[None, :, :, None, None] * ws[:, None]).sum(2)
        box = _box(H, W, dx, dy)
        return ws, box if case["box_forward"] else None, None if case["periodic"] else box

    U, Z = torch.zeros_like(x), torch.zeros_like(x)
    for s, (dx, dy, inv) in enumerate(rows):
        ws, fwd, mir = plane(s, dx, dy)
        wf = ws if fwd is None else ws * fwd
        U += wf * _at(x, dx, dy)
        Z += wf
        if inv:
            wm = ws if mir is None else ws * mir
            U += _back(wm * x, dx, dy)
            Z += _back(wm, dx, dy).expand_as(x)
    if case["op"] == "accumulate":
        got = {"U": U, "Z": Z}
        gU, gZ = (t["g0"].double(), t["g1"].double()) if case["train"] else (None, None)
    else:
        D = U / Z
        got = {"D": D, "log_C": Z.log()} if case["degree"] else {"D": D}
        if case["train"]:
            gD = t["g0"].double()
            gL = t["g1"].double() if case["degree"] else torch.zeros_like(gD)
            gU, gZ = gD / Z, (gL - gD * D) / Z
    if not case["train"]:
        return got
    gx = torch.zeros_like(x)
    gw = torch.empty(t["w"].shape, dtype=torch.float64, device=DEV)
    for s, (dx, dy, inv) in enumerate(rows):
        ws, fwd, mir = plane(s, dx, dy)
        wf = ws if fwd is None else ws * fwd
        gs = gU * _at(x, dx, dy) + gZ
        if fwd is not None:
            gs = gs * fwd
        gx += _back(wf * gU, dx, dy)
        if inv:
            gUn = _at(gU, dx, dy)
            gm = gUn * x + _at(gZ, dx, dy)
            wm = ws
            if mir is not None:
                gm, wm = gm * mir, ws * mir
            gs = gs + gm
            gx += wm * gUn
        if case["log"]:
            gs = gs * ws
        gw[s * B:(s + 1) * B] = gs.sum(1, keepdim=True) if case["shared"] else gs
    return {**got, "grad_x": gx, "grad_w": gw}


def _exact_metropolis(case, t, x, rows):
    """grad_w is left out: it is not continuous in the degrees (see
    ``tolerance``), so 64 bits do not say what 32 bits should give."""
    H, W = case["H"], case["W"]

    def plane(s, dx, dy):
        ws = t["w"][:, s].double()
        return ws * _box(H, W, dx, dy) if case["use_box"] else ws

    d = torch.zeros_like(x)
    for s, (dx, dy, inv) in enumerate(rows):
        ws = plane(s, dx, dy)
        d += ws
        if inv:
            d += _back(ws, dx, dy)
    K = {"x": torch.zeros_like(x), "e": torch.zeros_like(x), "g": torch.zeros_like(x)}
    vec = {"x": x, "e": torch.ones_like(x)}
    if case["train"]:
        vec["g"] = t["g0"].double()
    for s, (dx, dy, inv) in enumerate(rows):
        wk = plane(s, dx, dy) / torch.maximum(d, _at(d, dx, dy)).clamp_min(EPS)
        for k, v in vec.items():
            if k != "g":
                K[k] += wk * _at(v, dx, dy)
                if inv:
                    K[k] += _back(wk * v, dx, dy)
            else:  # the transpose
                K[k] += _back(wk * v, dx, dy)
                if inv:
                    K[k] += wk * _at(v, dx, dy)
    got = {"Wx": x - K["e"] * x + K["x"], "d_hat": K["e"]}
    if case["train"]:
        got["grad_x"] = vec["g"] * (1 - K["e"]) + K["g"]
        got["grad_w"] = None
    return got
