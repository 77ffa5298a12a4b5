"""The work whose speed this repository is judged by, as a program that uses it has it done.

A case is one training step (or one inference) of a single layer, through ``katsu_amd.ops`` on
device tensors: a convolution's forward and its one-call backward (dX and dW together, as
Katsu's ``backward_buffers`` computes them), or a matmul's forward and its VJP into fresh zero
buffers, as the autograd engine keeps them.  One case is a whole chain: the stem layer, its mean
pool and its matmul head, forward and backward.  All data are contiguous float32, the only type
the framework has; the sizes are those of its benchmark, its example and its tests, and common
ones between them.

``draw`` spreads over the same ranges: filters of 1, 3, 5 and 7, strides 1 and 2, from a few
channels to 512, images from 7 to 224 pixels wide, batches from 1 to 64, matrix sides from 16 to
4096, odd numbers among all of them.
"""
import math

import torch

from katsu_amd import ops

# Largest work of a drawn convolution pass: the stem layer's 15.1 GFLOP, and its 51 M output values.
MAX_CONV_FLOPS = 15.2e9
MAX_CONV_ELEMS = 52e6


def _conv(name, x, w, stride, pad, law="n01", mode="step"):
    n, c, h, wd = x
    k, _, r, s = w
    case = dict(kind="conv", mode=mode, n=n, c=c, h=h, w=wd, k=k, r=r, s=s, stride=stride,
                pad=pad, law=law)
    if name:
        case["name"] = name
    return case


def _matmul(name, m, k, n):
    case = dict(kind="matmul", m=m, k=k, n=n)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # The smallest calls.  Matrices of a toy program or a last layer, where launches are all:
        # the repository's own parity sizes.
        _matmul("matmul_small", 48, 40, 56),
        # The repository's example layer: one RGB image through eight 3x3 filters.
        _conv("example_layer", (1, 3, 224, 224), (8, 3, 3, 3), 1, 1, "u11"),
        # Inference of one image through one residual-block layer: forward only.
        _conv("infer_one_image", (1, 64, 56, 56), (64, 64, 3, 3), 1, 1, "u11", "forward"),
        # Matmul training steps: the benchmark's smallest and largest squares, and a ragged one
        # whose sides are multiples of nothing.
        _matmul("matmul_512", 512, 512, 512),
        _matmul("matmul_ragged", 1001, 1531, 777),
        _matmul("matmul_4096", 4096, 4096, 4096),
        # The benchmark's layers, batches of 32: a residual block's 3x3, and the two layers that
        # halve the image (3x3 and 1x1, stride 2).
        _conv("resnet_3x3", (32, 64, 56, 56), (64, 64, 3, 3), 1, 1, "u11"),
        _conv("down_3x3", (32, 128, 28, 28), (256, 128, 3, 3), 2, 1),
        _conv("down_1x1", (32, 128, 28, 28), (256, 128, 1, 1), 2, 0),
        # A deep layer of the same network family: many channels on small images.
        _conv("deep_3x3", (32, 256, 14, 14), (256, 256, 3, 3), 1, 1),
        # A layer of a program that does not choose round numbers: odd image sides and channel
        # counts, a 5x5 filter.
        _conv("ragged_5x5", (7, 45, 37, 51), (83, 45, 5, 5), 1, 2),
        # The benchmark's stem chain: 7x7 stride-2 convolution of 64 images, mean pool, matmul
        # head of 1000 classes, and the way back to the image and the filters.
        dict(name="stem_chain", kind="chain", n=64, c=3, h=224, w=224, k=64, r=7, s=7, stride=2,
             pad=3, law="u01", classes=1000),
    ]


def _log_int(rng, lo, hi):
    """An integer in [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _round_or_not(rng, v, step, lo):
    """v as it is (odd sizes among them), or rounded to a multiple of step."""
    return v if rng.random() < 0.5 else max(lo, step * ((v + step // 2) // step))


def draw(rng):
    if rng.random() < 0.4:
        m, k, n = (_round_or_not(rng, _log_int(rng, 16, 4096), 16, 16) for _ in range(3))
        return _matmul(None, m, k, n)
    while True:
        f, st = rng.choice([(1, 1), (1, 2), (3, 1), (3, 1), (3, 2), (5, 1), (5, 2), (7, 2)])
        n = _log_int(rng, 1, 64)
        c = _log_int(rng, 3, 512)
        c = _round_or_not(rng, c, 16, 16) if c > 8 else c
        k = _round_or_not(rng, _log_int(rng, 8, 512), 16, 16)
        h = _log_int(rng, 7, 224)
        w = h if rng.random() < 0.6 else _log_int(rng, max(7, h // 2), min(224, 2 * h))
        mode = "forward" if rng.random() < 0.2 else "step"
        case = _conv(None, (n, c, h, w), (k, c, f, f), st, f // 2, "n01", mode)
        oh, ow = _out(case)
        if (_conv_flops(case) <= MAX_CONV_FLOPS and n * k * oh * ow <= MAX_CONV_ELEMS
                and n * c * h * w <= MAX_CONV_ELEMS):
            return case


def _out(case):
    return ((case["h"] + 2 * case["pad"] - case["r"]) // case["stride"] + 1,
            (case["w"] + 2 * case["pad"] - case["s"]) // case["stride"] + 1)


def _conv_flops(case):
    """FLOP of one pass (forward, dX or dW), padding counted."""
    oh, ow = _out(case)
    return 2.0 * case["n"] * case["k"] * oh * ow * case["c"] * case["r"] * case["s"]


# ---- inputs ---------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _image(gen, shape, law):
    """Pixels in [0, 1), values in [-1, 1), or unit-variance activations."""
    if law == "n01":
        return torch.randn(shape, generator=gen, device="cuda")
    x = torch.rand(shape, generator=gen, device="cuda")
    return x if law == "u01" else x.mul_(2).sub_(1)


def _inputs(case, seed):
    gen = _gen(seed)
    if case["kind"] == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        a = _image(gen, (m, k), "u11")
        b = _image(gen, (k, n), "u11")
        return a, b, torch.randn((m, n), generator=gen, device="cuda")
    n, c, h, w = case["n"], case["c"], case["h"], case["w"]
    k, r, s = case["k"], case["r"], case["s"]
    oh, ow = _out(case)
    x = _image(gen, (n, c, h, w), case["law"])
    # He initialisation, as the framework's seeded layers have it.
    wt = torch.randn((k, c, r, s), generator=gen, device="cuda") * math.sqrt(2.0 / (c * r * s))
    if case["kind"] == "chain":
        head = torch.randn((k, case["classes"]), generator=gen, device="cuda") * math.sqrt(2.0 / k)
        glog = torch.randn((n, case["classes"]), generator=gen, device="cuda") / n
        return x, wt, head, glog
    gy = torch.randn((n, k, oh, ow), generator=gen, device="cuda")
    return x, wt, gy


def prepare(case, seed):
    st = {"case": dict(case), "in": _inputs(case, seed)}
    new = lambda *shape: torch.empty(shape, device="cuda")
    if case["kind"] == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        st.update(c=new(m, n), da=new(m, k), db=new(k, n))
        return st
    n, k = case["n"], case["k"]
    oh, ow = _out(case)
    x, wt = st["in"][0], st["in"][1]
    st["y"] = new(n, k, oh, ow)
    if case.get("mode") != "forward":
        st.update(dx=torch.empty_like(x), dw=torch.empty_like(wt))
    if case["kind"] == "chain":
        cl = case["classes"]
        st.update(p=new(n * k), logits=new(n, cl), dp=new(n, k), dhead=new(k, cl),
                  dy=new(n, k, oh, ow))
    return st


# ---- one pass -------------------------------------------------------------------------------

def run(st):
    case = st["case"]
    if case["kind"] == "matmul":
        a, b, g = st["in"]
        m, k, n = case["m"], case["k"], case["n"]
        ops.gemm(a, b, m, n, k, out=st["c"])
        ops.fill(st["da"], 0.0)
        ops.fill(st["db"], 0.0)
        ops.matmul_vjp(a, b, g, st["da"], st["db"])
        return {"c": st["c"], "da": st["da"], "db": st["db"]}
    stride, pad = case["stride"], case["pad"]
    if case["kind"] == "conv":
        x, wt, gy = st["in"]
        ops.conv2d_forward(x, wt, stride, pad, out=st["y"])
        if case["mode"] == "forward":
            return {"y": st["y"]}
        ops.conv2d_backward(x, wt, gy, stride, pad, dx=st["dx"], dw=st["dw"])
        return {"y": st["y"], "dx": st["dx"], "dw": st["dw"]}
    x, wt, head, glog = st["in"]
    n, k, cl = case["n"], case["k"], case["classes"]
    oh, ow = _out(case)
    ops.conv2d_forward(x, wt, stride, pad, out=st["y"])
    ops.mean_rows(st["y"], n * k, oh * ow, out=st["p"])
    p = st["p"].view(n, k)
    ops.gemm(p, head, n, cl, k, out=st["logits"])
    ops.fill(st["dp"], 0.0)
    ops.fill(st["dhead"], 0.0)
    ops.matmul_vjp(p, head, glog, st["dp"], st["dhead"])
    ops.broadcast_rows(st["dp"], n * k, oh * ow, 1.0 / (oh * ow), dy=st["dy"])
    ops.conv2d_backward(x, wt, st["dy"], stride, pad, dx=st["dx"], dw=st["dw"])
    return {"logits": st["logits"], "dhead": st["dhead"], "dx": st["dx"], "dw": st["dw"]}


# ---- what a pass cannot do without -------------------------------------------------------------

def work(case):
    if case["kind"] == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        # a, b and g read once, c, da and db written once; three products.
        return {"bytes": 4.0 * 2 * (m * k + k * n + m * n), "flops": 6.0 * m * k * n}
    oh, ow = _out(case)
    nx = case["n"] * case["c"] * case["h"] * case["w"]
    nw = case["k"] * case["c"] * case["r"] * case["s"]
    ny = case["n"] * case["k"] * oh * ow
    f = _conv_flops(case)
    if case["kind"] == "conv":
        if case["mode"] == "forward":
            return {"bytes": 4.0 * (nx + nw + ny), "flops": f}
        return {"bytes": 4.0 * 2 * (nx + nw + ny), "flops": 3 * f}
    # The chain reads x twice (the forward and the filter gradient stand a whole head apart) and
    # writes dx; y and dy are its own, but no call it makes can do without either: each is
    # written once and read once.
    nh = case["k"] * case["classes"]
    nl = case["n"] * case["classes"]
    return {"bytes": 4.0 * (3 * nx + 2 * nw + 4 * ny + 2 * nh + 2 * nl),
            "flops": 3 * f + 6.0 * case["n"] * nh}


def tolerance(case):
    """Four times the largest error against float64 that the outputs showed in the 2-norm: 1.1e-6
    over the listed cases and 1.6e-6 over twenty drawn ones.  It is the rounding of float32 sums,
    which grows slowly with their length."""
    return {"rel": 6e-6}


# ---- the same in float64 -------------------------------------------------------------------------

def _taps(case):
    oh, ow = _out(case)
    st = case["stride"]
    for i in range(case["r"]):
        for j in range(case["s"]):
            yield i, j, slice(i, i + st * (oh - 1) + 1, st), slice(j, j + st * (ow - 1) + 1, st)


def _exact_forward(case, x, wt):
    oh, ow = _out(case)
    p = case["pad"]
    xp = torch.nn.functional.pad(x, (p, p, p, p))
    y = torch.zeros((case["n"], case["k"], oh * ow), device=x.device, dtype=x.dtype)
    for i, j, rows, cols in _taps(case):
        xs = xp[:, :, rows, cols].reshape(case["n"], case["c"], oh * ow)
        y += torch.matmul(wt[:, :, i, j].contiguous(), xs)
    return y.view(case["n"], case["k"], oh, ow)


def _exact_backward(case, x, wt, gy):
    oh, ow = _out(case)
    n, c, k, p = case["n"], case["c"], case["k"], case["pad"]
    h, w = case["h"], case["w"]
    xp = torch.nn.functional.pad(x, (p, p, p, p))
    dxp = torch.zeros_like(xp)
    dw = torch.empty_like(wt)
    g = gy.reshape(n, k, oh * ow)
    gk = g.transpose(0, 1).reshape(k, n * oh * ow).contiguous()
    for i, j, rows, cols in _taps(case):
        xs = xp[:, :, rows, cols].reshape(n, c, oh * ow)
        xc = xs.transpose(0, 1).reshape(c, n * oh * ow).t().contiguous()
        dw[:, :, i, j] = torch.matmul(gk, xc)
        dxp[:, :, rows, cols] += torch.matmul(wt[:, :, i, j].t().contiguous(),
                                              g).view(n, c, oh, ow)
    return dxp[:, :, p:p + h, p:p + w].contiguous(), dw


def exact(case, seed):
    ins = [t.double() for t in _inputs(case, seed)]
    if case["kind"] == "matmul":
        a, b, g = ins
        return {"c": torch.matmul(a, b), "da": torch.matmul(g, b.t().contiguous()),
                "db": torch.matmul(a.t().contiguous(), g)}
    if case["kind"] == "conv":
        x, wt, gy = ins
        y = _exact_forward(case, x, wt)
        if case["mode"] == "forward":
            return {"y": y}
        dx, dw = _exact_backward(case, x, wt, gy)
        return {"y": y, "dx": dx, "dw": dw}
    x, wt, head, glog = ins
    n, k = case["n"], case["k"]
    oh, ow = _out(case)
    y = _exact_forward(case, x, wt)
    p = y.reshape(n * k, oh * ow).mean(dim=1).view(n, k)
    dp = torch.matmul(glog, head.t().contiguous())
    dy = (dp / (oh * ow)).view(n, k, 1, 1).expand(n, k, oh, ow).contiguous()
    dx, dw = _exact_backward(case, x, wt, dy)
    return {"logits": torch.matmul(p, head), "dhead": torch.matmul(p.t().contiguous(), glog),
            "dx": dx, "dw": dw}
