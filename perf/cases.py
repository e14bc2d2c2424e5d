"""Performance cases of the transform library on one GPU.

Each case is one pass of work as a user's program does it, through the
package's public entry points, on device arrays:

  pair    forward then backward 3-d transform (c2c, or r2c then c2r), out of
          place: pseudo-spectral codes, convolution and Poisson solvers
  ousam   oversampled, shifted r2c forward and its adjoint through autograd:
          non-uniform FFTs and gradient-based reconstruction
  r2r     DCT-II then DCT-III: solvers with Neumann boundaries
  batch   many independent c2c transforms of different sizes in one call
  ghost   ghost-cell exchange of one field and reduce of another:
          particle-mesh interpolation and charge assignment

listed() names the representative cases, draw() takes further ones from the
same ranges, prepare()/run() execute one, work() is the data and arithmetic
a pass cannot do without, exact() the result in 64-bit arithmetic by plain
torch.
"""
import math

import torch

import pfft_amd as P
from pfft_amd.autograd import apply_plan

DEV = "cuda:0"
BATCH_SIDES = (24, 32, 48, 60, 64, 80, 96, 128)


# ---------------------------------------------------------------- cases
def listed():
    return [
        # the parity suite's uneven size, transposed layouts: a tiny grid
        # inside a time step, where latency and launches are all there is
        _pair("uneven-29x27x31-f64", "c2c", [29, 27, 31], "f64", transposed=True),
        # the smallest benchmark configuration, default layout
        _pair("c2c-64-f64", "c2c", [64, 64, 64], "f64"),
        # a vector field (three interleaved components) on an ordinary grid
        _pair("vector-r2c-128x3-f64", "r2c", [128, 128, 128], "f64", howmany=3),
        # single-precision spectral step on an ordinary grid
        _pair("r2c-256-f32", "r2c", [256, 256, 256], "f32", transposed=True),
        # the headline benchmark: 512^3 r2c TRANSPOSED_OUT, c2r TRANSPOSED_IN
        _pair("r2c-512-f64", "r2c", [512, 512, 512], "f64", transposed=True),
        # the mixed-precision form of a large complex grid
        _pair("c2c-512-bf16x2", "c2c", [512, 512, 512], "f32", form="bf16x2"),
        # grid sides chosen by the physics, not by the FFT: smooth but not a
        # power of two, and with factors beyond 2, 3 and 5
        _pair("c2c-360x300x250-f64", "c2c", [360, 300, 250], "f64"),
        _pair("r2c-210x196x330-f32", "r2c", [210, 196, 330], "f32", transposed=True),
        # oversampled shifted transform and its gradient (128^3 -> 256^3)
        {"name": "ousam-128-256-f32", "family": "ousam", "ni": 128, "n": 256, "prec": "f32"},
        # DCT pair of a Neumann problem
        {"name": "dct-256-f64", "family": "r2r", "n0": 256, "n1": 256, "n2": 256,
         "prec": "f64"},
        # 384 uneven complex64 transforms, sides 24..128, in one call
        {"name": "batch-384-f32", "family": "batch", "count": 384, "sizes_seed": 20261202,
         "prec": "f32"},
        # ghost cells of a particle-mesh field: 256^3, 4 cells per side
        {"name": "ghost-256-f64", "family": "ghost", "n0": 256, "n1": 256, "n2": 256,
         "cells": 4, "prec": "f64"},
    ]


def _pair(name, kind, n, prec, transposed=False, howmany=1, form=""):
    return {"name": name, "family": "pair", "kind": kind, "n0": n[0], "n1": n[1], "n2": n[2],
            "prec": prec, "transposed": transposed, "howmany": howmany, "form": form}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(rng, lo, hi, primes=(2, 3, 5, 7)):
    """a length near a log-uniform target with prime factors from `primes`"""
    m = _log_int(rng, lo, hi)
    while True:
        r = m
        for q in primes:
            while r % q == 0:
                r //= q
        if r == 1:
            return m
        m -= 1


def _side(rng, lo, hi):
    """one grid side: a power of two, a smooth number or any number"""
    u = rng.random()
    if u < 0.35:
        return 1 << rng.randint(math.ceil(math.log2(lo)), math.floor(math.log2(hi)))
    if u < 0.75:
        return _smooth(rng, lo, hi)
    return _log_int(rng, lo, min(hi, 160))


def draw(rng):
    u = rng.random()
    prec = rng.choice(("f64", "f32"))
    if u < 0.6:
        kind = rng.choice(("c2c", "r2c"))
        howmany = rng.choice((1, 1, 1, 1, 2, 3))
        form = ""
        while True:
            n = [_side(rng, 16, 1024) for _ in range(3)]
            pow2 = all(v & (v - 1) == 0 for v in n)
            cap = (1 << 26) if pow2 else (1 << 23)
            if n[0] * n[1] * n[2] * howmany <= cap:
                break
        if kind == "c2c" and prec == "f32" and pow2 and howmany == 1:
            form = rng.choice(("", "f32mfma", "bf16x2"))
        c = _pair("", kind, n, prec, transposed=rng.random() < 0.5, howmany=howmany, form=form)
        del c["name"]
        return c
    if u < 0.7:
        n = 2 * _smooth(rng, 24, 144, (2, 3, 5))
        ni = 2 * max(4, int(n / 2 / rng.uniform(1.2, 2.0)))
        return {"family": "ousam", "ni": ni, "n": n, "prec": prec}
    if u < 0.8:
        n = [_smooth(rng, 16, 384) for _ in range(3)]
        while n[0] * n[1] * n[2] > 1 << 23:
            n[n.index(max(n))] //= 2
        return {"family": "r2r", "n0": n[0], "n1": n[1], "n2": n[2], "prec": prec}
    if u < 0.9:
        return {"family": "batch", "count": _log_int(rng, 4, 256),
                "sizes_seed": rng.randint(1, 1 << 30), "prec": prec}
    return {"family": "ghost", "n0": _log_int(rng, 24, 256), "n1": _log_int(rng, 24, 256),
            "n2": _log_int(rng, 24, 256), "cells": rng.randint(1, 6), "prec": prec}


# ---------------------------------------------------------------- helpers
def _n(case):
    return [case["n0"], case["n1"], case["n2"]]


def _dtypes(prec):
    return (torch.float64, torch.complex128) if prec == "f64" else (torch.float32, torch.complex64)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(shape, dtype, seed):
    return torch.randn(shape, generator=_gen(seed), device=DEV, dtype=dtype)


def _mesh():
    rc, comm = P.create_procmesh([1, 1])
    assert rc == 0
    return comm


def _batch_sizes(case):
    g = torch.Generator().manual_seed(case["sizes_seed"])
    idx = torch.randint(len(BATCH_SIDES), (case["count"], 3), generator=g)
    return [[BATCH_SIDES[i] for i in row] for row in idx.tolist()]


def _batch_inputs(case, seed):
    """one array holding every input back to back, and views of it"""
    sizes = _batch_sizes(case)
    cdt = _dtypes(case["prec"])[1]
    flat = _randn((sum(a * b * c for a, b, c in sizes),), cdt, seed)
    return sizes, flat, _views(flat, sizes)


def _views(flat, sizes):
    out, o = [], 0
    for a, b, c in sizes:
        out.append(flat[o:o + a * b * c].view(a, b, c))
        o += a * b * c
    return out


def _pair_input(case, seed):
    rdt, cdt = _dtypes(case["prec"])
    shape = _n(case) + ([case["howmany"]] if case["howmany"] > 1 else [])
    return _randn(shape, rdt if case["kind"] == "r2c" else cdt, seed)


def _ghost_inputs(case, seed):
    """a field (block) and deposited charge (box with its ghost cells)"""
    rdt = _dtypes(case["prec"])[0]
    n, c = _n(case), case["cells"]
    return _randn(n, rdt, seed), _randn([v + 2 * c for v in n], rdt, seed + 1)


# ---------------------------------------------------------------- prepare
def prepare(case, seed):
    state = globals()["_prepare_" + case["family"]](case, seed)
    state["run"] = globals()["_run_" + case["family"]]
    torch.cuda.synchronize()     # the library runs on its own stream
    return state


def _prepare_pair(case, seed):
    rdt, cdt = _dtypes(case["prec"])
    n, h = _n(case), case["howmany"]
    x = _pair_input(case, seed)
    k = list(n)
    if case["kind"] == "r2c":
        k[2] = n[2] // 2 + 1
    if case["transposed"]:
        k = [k[1], k[2], k[0]]
    k = torch.empty(k + ([h] if h > 1 else []), dtype=cdt, device=DEV)
    y = torch.empty_like(x)
    comm = _mesh()
    form = {"": 0, "f32mfma": P.AMD_MFMA_F32, "bf16x2": P.AMD_MFMA_BF16X2}[case["form"]]
    back = "c2r" if case["kind"] == "r2c" else "c2c"
    fw = P.Plan(case["kind"], n, x.data_ptr(), k.data_ptr(), howmany=h, sign=P.FORWARD,
                flags=form | (P.TRANSPOSED_OUT if case["transposed"] else 0), comm=comm,
                prec=case["prec"])
    bw = P.Plan(back, n, k.data_ptr(), y.data_ptr(), howmany=h, sign=P.BACKWARD,
                flags=form | (P.TRANSPOSED_IN if case["transposed"] else 0), comm=comm,
                prec=case["prec"])
    assert fw.ok and bw.ok
    return {"x": x, "k": k, "y": y, "fw": fw, "bw": bw}


def _run_pair(s):
    s["fw"].execute()
    s["bw"].execute()
    return s["k"], s["y"]


def _prepare_ousam(case, seed):
    rdt, cdt = _dtypes(case["prec"])
    ni, n = case["ni"], case["n"]
    x = _randn([ni] * 3, rdt, seed)
    g = _randn([n, n, n // 2 + 1], cdt, seed + 1)
    k = torch.empty_like(g)
    plan = P.Plan("r2c", [n] * 3, x.data_ptr(), k.data_ptr(), ni=[ni] * 3,
                  flags=P.SHIFTED_IN | P.SHIFTED_OUT, comm=_mesh(), prec=case["prec"])
    assert plan.ok
    return {"x": x.requires_grad_(True), "g": g, "plan": plan, "k": k}


def _run_ousam(s):
    X = apply_plan(s["x"], s["plan"], tuple(s["g"].shape), True)
    gx, = torch.autograd.grad(X, s["x"], s["g"])
    return X.detach(), gx


def _prepare_r2r(case, seed):
    rdt = _dtypes(case["prec"])[0]
    n = _n(case)
    x = _randn(n, rdt, seed)
    k, y = torch.empty_like(x), torch.empty_like(x)
    comm = _mesh()
    fw = P.Plan("r2r", n, x.data_ptr(), k.data_ptr(), comm=comm, prec=case["prec"],
                kinds=[P.REDFT10] * 3)
    bw = P.Plan("r2r", n, k.data_ptr(), y.data_ptr(), comm=comm, prec=case["prec"],
                kinds=[P.REDFT01] * 3)
    assert fw.ok and bw.ok
    return {"x": x, "k": k, "y": y, "fw": fw, "bw": bw}


_run_r2r = _run_pair


def _prepare_batch(case, seed):
    sizes, flat, xs = _batch_inputs(case, seed)
    out = torch.empty_like(flat)
    comm = _mesh()
    plans = [P.Plan("c2c", n, x.data_ptr(), y.data_ptr(), comm=comm, prec=case["prec"])
             for n, x, y in zip(sizes, xs, _views(out, sizes))]
    assert all(p.ok for p in plans)
    return {"in": flat, "out": out, "plans": plans}


def _run_batch(s):
    P.execute_batch(s["plans"])
    return s["out"]


def _prepare_ghost(case, seed):
    n, c = _n(case), case["cells"]
    field, charge = _ghost_inputs(case, seed)
    comm = _mesh()
    s = {"field": field, "charge": charge, "n": n}
    for name in ("exg", "red"):
        box = torch.empty([v + 2 * c for v in n], dtype=field.dtype, device=DEV)
        plan = P.GcPlan("r", n, box.data_ptr(), [c] * 3, [c] * 3, comm=comm, prec=case["prec"])
        assert plan.ok
        s[name], s[name + "_plan"] = box, plan
    return s


def _run_ghost(s):
    # the arrays are worked on in place: the program writes its data into them first
    s["exg"].view(-1)[:s["field"].numel()].copy_(s["field"].view(-1))
    s["red"].copy_(s["charge"])
    torch.cuda.current_stream().synchronize()
    s["exg_plan"].exchange()
    s["red_plan"].reduce()
    return s["exg"], s["red"]


def run(state):
    return state["run"](state)


# ---------------------------------------------------------------- work
def work(case):
    es = 8 if case["prec"] == "f64" else 4
    fam = case["family"]
    if fam == "ghost":
        n = _n(case)
        block = n[0] * n[1] * n[2]
        box = 1
        for v in n:
            box *= v + 2 * case["cells"]
        # both fills (read, write), exchange (block -> box), reduce (box -> box)
        return {"bytes": es * (2 * block + 2 * box + block + box + 2 * box), "flops": box - block}
    if fam == "batch":
        pts = [a * b * c for a, b, c in _batch_sizes(case)]
        return {"bytes": 2 * 2 * es * sum(pts), "flops": sum(5 * v * math.log2(v) for v in pts)}
    if fam == "ousam":
        n, ni = case["n"], case["ni"]
        spec = 2 * n * n * (n // 2 + 1)
        return {"bytes": 2 * es * (ni ** 3 + spec), "flops": 5.0 * n ** 3 * math.log2(n ** 3)}
    n = _n(case)
    pts = n[0] * n[1] * n[2]
    if fam == "r2r":
        return {"bytes": 4 * es * pts, "flops": 5.0 * pts * math.log2(pts)}
    h = case["howmany"]
    if case["kind"] == "c2c":
        return {"bytes": 4 * 2 * es * pts * h, "flops": 10.0 * pts * h * math.log2(pts)}
    spec = 2 * n[0] * n[1] * (n[2] // 2 + 1)
    return {"bytes": 2 * es * (pts + spec) * h, "flops": 5.0 * pts * h * math.log2(pts)}


# ---------------------------------------------------------------- exact
def exact(case, seed):
    return globals()["_exact_" + case["family"]](case, seed)


def _exact_pair(case, seed):
    x = _pair_input(case, seed)
    n = _n(case)
    x = x.to(torch.float64 if case["kind"] == "r2c" else torch.complex128)
    y = x * float(n[0] * n[1] * n[2])
    k = (torch.fft.rfftn if case["kind"] == "r2c" else torch.fft.fftn)(x, dim=(0, 1, 2))
    if case["transposed"]:
        k = k.permute([1, 2, 0] + ([3] if case["howmany"] > 1 else []))
    return k.contiguous(), y


def _exact_ousam(case, seed):
    rdt, cdt = _dtypes(case["prec"])
    ni, n = case["ni"], case["n"]
    o = (n - ni) // 2
    cut = slice(n // 2 - ni // 2, n // 2 - ni // 2 + ni)
    assert cut.start == o
    x = _randn([ni] * 3, rdt, seed).double()
    g = _randn([n, n, n // 2 + 1], cdt, seed + 1).to(torch.complex128)
    # centred transform of the zero-padded cube, l2 in [-n/2, 0] kept
    xe = torch.zeros([n] * 3, dtype=torch.complex128, device=DEV)
    xe[cut, cut, cut] = x.to(torch.complex128)
    X = torch.fft.fftshift(torch.fft.fftn(torch.fft.ifftshift(xe)))[:, :, :n // 2 + 1]
    # the adjoint: Re sum_l g_l exp(+2 pi i j l / n)
    ge = torch.zeros([n] * 3, dtype=torch.complex128, device=DEV)
    ge[:, :, :n // 2 + 1] = g
    gx = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(ge), norm="forward"))
    return X.contiguous(), gx[cut, cut, cut].real.contiguous()


def _dct2(x, dim):
    """FFTW's REDFT10 along one dimension: 2 sum_j x_j cos(pi (j+1/2) k / n)"""
    n = x.shape[dim]
    k = torch.arange(n, device=DEV, dtype=torch.int64)
    arg = (2 * k[None, :] + 1) * k[:, None] % (4 * n)
    c = 2 * torch.cos(arg.double() * (math.pi / (2 * n)))
    return torch.movedim(torch.movedim(x, dim, -1).contiguous() @ c.t().contiguous(), -1, dim)


def _exact_r2r(case, seed):
    n = _n(case)
    x = _randn(n, _dtypes(case["prec"])[0], seed).double()
    k = x
    for d in range(3):
        k = _dct2(k, d)
    return k.contiguous(), x * float(8 * n[0] * n[1] * n[2])


def _exact_batch(case, seed):
    xs = _batch_inputs(case, seed)[2]
    return torch.cat([torch.fft.fftn(x.cpu().to(torch.complex128)).view(-1) for x in xs]).to(DEV)


def _exact_ghost(case, seed):
    n, c = _n(case), case["cells"]
    field, charge = _ghost_inputs(case, seed)
    own = [(torch.arange(v + 2 * c, device=DEV) - c) % v for v in n]
    box = field.double()[own[0][:, None, None], own[1][None, :, None], own[2][None, None, :]]
    red = charge.double()
    for d in range(3):
        shape = list(red.shape)
        shape[d] = n[d]
        red = torch.zeros(shape, dtype=torch.float64, device=DEV).index_add_(d, own[d], red)
    out = torch.zeros(charge.numel(), dtype=torch.float64, device=DEV)
    out[:red.numel()] = red.view(-1)
    return box, out.view(charge.shape)
