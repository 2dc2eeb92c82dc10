"""The work that programs have this library do, as cases to time.

Every case goes through the public entry points (prodm_amd.mdr, .batched,
.autograd and the C ABI under them) with the inputs such a program holds on
the GPU, and returns what the call leaves behind: plane words, level tables,
coefficients, gradients, reconstructed fields. Grid extents are m 2^L + 1,
the extents that L levels accept; m is odd in the ragged cases.

kinds
    step       refactor a resident field, retrieve it again (one Plan)
    batch      one refactor of several uneven fields (Batch)
    transform  MGARD decompose and recompose alone
    gradient   recompose forward and its transpose (torch.autograd)
    composed   the refactor / reconstruct loop built from the components
    tables     level-error tables of one level's coefficients
    streams    plane streams to host bytes and back, then a retrieve
    codec      bitplane encode (and decode) of one level's coefficients
"""
import ctypes as C
import math
import random

import numpy as np
import torch

from prodm_amd import autograd, batched, capi, mdr

_DT = {"f32": torch.float32, "f64": torch.float64}
_ENC = {"negabinary": capi.NEGABINARY, "grouped": capi.GROUPED, "perbit": capi.PERBIT}


def _case(kind, dims, L, dtype="f32", nb=32, encoder="negabinary", **more):
    return {"kind": kind, "dims": "x".join(str(d) for d in dims), "L": L, "dtype": dtype, "nb": nb,
            "encoder": encoder, **more}


def listed():
    return [
        # the smallest call: a 33^3 block, every plane read back; launches and their gaps
        dict(_case("step", [33] * 3, 3), name="step_33", graph=False, hier=False, full=True),
        # the ordinary one: 129^3 simulation output, GroupedBP streams
        dict(_case("step", [129] * 3, 4, encoder="grouped"), name="step_129_grouped", graph=False, hier=False,
             full=False),
        # bench.py's workload: 513^3 float32, replayed from the plan's graphs
        dict(_case("step", [513] * 3, 6), name="step_513_graph", graph=True, hier=False, full=False),
        # the largest: an anisotropic float64 turbulence field, 64 planes
        dict(_case("step", [1025, 1025, 257], 7, "f64", 64, "grouped"), name="step_1025_f64_grouped", graph=False,
             hier=False, full=False),
        # hierarchical basis with PerBit streams (decoded on the host), as the GE applications pair them
        dict(_case("step", [129] * 3, 4, encoder="perbit"), name="step_129_perbit", graph=False, hier=True, full=False),
        # a dozen variables of uneven shapes, written out together
        dict(_case("batch", [0], 4), name="batch_12", fields=12, shapes=3),
        # a ragged 2-D float64 grid through the transform alone
        dict(_case("transform", [1537, 769], 6, "f64"), name="transform_1537x769_f64", hier=False),
        # sensitivities of a quantity of interest: forward and backward at 257^3
        dict(_case("gradient", [257] * 3, 5), name="gradient_257"),
        # a ragged field through the component loop (the drop-in for ProDM's composers)
        dict(_case("composed", [353, 161, 97], 5), name="composed_353x161x97"),
        # error tables of the finest level of a 257^3 field
        dict(_case("tables", [257 ** 3 - 129 ** 3], 0), name="tables_257"),
        # streams out to host memory and back in, plane by plane
        dict(_case("streams", [129] * 3, 4), name="streams_129"),
        # PerBit encode of the finest level of a 513^3 field
        dict(_case("codec", [513 ** 3 - 257 ** 3], 0, encoder="perbit"), name="codec_perbit_513"),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _grid(rng, points, nd, L):
    """nd extents m 2^L + 1, uneven, about `points` nodes in all (never more than twice)"""
    w = [rng.uniform(-0.6, 0.6) for _ in range(nd)]
    side = [points ** (1.0 / nd) * math.exp(x - sum(w) / nd) for x in w]
    return [max(1, int(s / 2 ** L)) * 2 ** L + 1 for s in side]


def draw(rng):
    kind = rng.choice(["step", "step", "step", "batch", "transform", "gradient", "composed", "tables", "streams",
                       "codec", "codec"])
    dtype = rng.choice(["f32", "f32", "f64"])
    nb = 32 if dtype == "f32" else 64
    if kind == "batch":
        return _case(kind, [0], 4, fields=rng.randint(3, 12), shapes=rng.randint(10, 1 << 20))
    if kind == "tables":
        return _case(kind, [int(_log_uniform(rng, 3e3, 3e7))], 0)
    if kind == "codec":
        encoder = rng.choice(["negabinary", "grouped", "perbit"])
        n = int(_log_uniform(rng, 3e3, 1e8 if dtype == "f32" else 3e7))
        return _case(kind, [n], 0, dtype, nb, encoder)
    nd = rng.choice([2, 3, 3, 3])
    most = {"step": 6e7, "transform": 6e7, "gradient": 1.7e7, "composed": 3e7, "streams": 2e6}[kind]
    if kind == "step":
        encoder = rng.choice(["negabinary", "negabinary", "grouped", "perbit"])
        points = _log_uniform(rng, 2e4, 1e6 if encoder == "perbit" else most / (1 if dtype == "f32" else 2))
    else:
        encoder = rng.choice(["negabinary", "grouped"]) if kind == "streams" else "negabinary"
        points = _log_uniform(rng, 2e4, most / (1 if dtype == "f32" else 2))
    L = rng.randint(2, max(2, min(7, int(math.log2(points ** (1.0 / nd))) - 2)))
    more = {}
    if kind == "step":
        more = {"graph": encoder != "perbit" and rng.random() < 0.4, "hier": rng.random() < 0.25,
                "full": rng.random() < 0.3}
    if kind == "transform":
        more = {"hier": rng.random() < 0.3}
    return _case(kind, _grid(rng, points, nd, L), L, dtype, nb, encoder, **more)


# ---- inputs ---------------------------------------------------------------
def _dims(case):
    return [int(d) for d in case["dims"].split("x")]


def _batch_shapes(case):
    """per field 2-D or 3-D, extents 2^k + 1, k in 5..9, at most 2^25 nodes"""
    rng = random.Random(case["shapes"])
    out = []
    for _ in range(case["fields"]):
        nd = rng.randint(2, 3)
        while True:
            dims = [2 ** rng.randint(5, 9) + 1 for _ in range(nd)]
            if math.prod(dims) <= 2 ** 25:
                break
        out.append(dims)
    return out


def _field(dims, dtype, seed):
    """a wave, Gaussian bumps and a little noise on the unit box (dense, dims[0] slowest)"""
    rng = np.random.default_rng(seed)
    nd = len(dims)
    ax = [torch.linspace(0.0, 1.0, n, dtype=torch.float64, device="cuda").view([-1 if k == d else 1 for k in range(nd)])
          for d, n in enumerate(dims)]
    amp, wid, mid = rng.uniform(0.5, 2.0, 8), rng.uniform(0.02, 0.1, 8), rng.uniform(0.0, 1.0, (8, nd))
    parts = [torch.sin(2 * math.pi * f * x + p) for f, x, p in zip((3, 5, 2), ax, rng.uniform(0, 6.28, nd))]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    u = torch.randn(dims, dtype=_DT[dtype], device="cuda", generator=gen)
    u *= 1e-4 if dtype == "f32" else 1e-8
    u += _product(parts)
    for b in range(8):
        u += amp[b] * _product([torch.exp(-((x - mid[b, d]) ** 2) / (2 * wid[b] ** 2)) for d, x in enumerate(ax)])
    return u.reshape(-1)


def _product(ts):
    p = ts[0]
    for t in ts[1:]:
        p = p * t
    return p


def _coefficients(n, dtype, seed):
    """multilevel coefficients: most of them orders of magnitude below the largest, some zero"""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    x = torch.randn(n, dtype=_DT[dtype], device="cuda", generator=gen)
    x *= torch.exp(1.5 * torch.randn(n, dtype=_DT[dtype], device="cuda", generator=gen) - 6.0)
    x[torch.rand(n, device="cuda", generator=gen) < 0.02] = 0
    return x


def _planes_read(L, nb, full):
    """planes per level of a retrieval: all of them, or fewer on the finer levels, as the greedy planner picks"""
    if full:
        return [nb] * (L + 1)
    return [nb - min(nb // 2 + nb // 8, (nb // 8) * max(0, l - 1)) for l in range(L + 1)]


class _Window:
    """a library-owned device buffer, for torch.as_tensor (no copy)"""

    def __init__(self, ptr, shape, strides, typestr):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "strides": strides,
                                         "typestr": typestr, "version": 3}


def _window(plan, ptr, shape, typestr, strides=None):
    t = torch.as_tensor(_Window(ptr, shape, strides, typestr), device="cuda")
    t.plan = plan  # the plan owns the memory: it lives as long as the tensor does
    return t


def _plane_windows(plan):
    """per level the plane words (planes, words) in the plan's storage; NegaBinary plans"""
    item = 4 if plan.dtype == torch.float32 else 8
    out = []
    for l in range(plan.L + 1):
        first, nbytes = plan.plane(l, 0)
        pitch = plan.plane(l, 1)[0] - first
        out.append(_window(plan, first, (plan.nb, nbytes // item), f"<i{item}", (pitch, item)))
    return out


def _level_windows(plan):
    """per level the interleaved coefficients in the plan's storage"""
    item = 4 if plan.dtype == torch.float32 else 8
    out = []
    for l in range(plan.L + 1):
        ptr = C.c_void_p()
        capi.check(capi.lib().prodm_mdr_level_coefficients(plan.h, l, C.byref(ptr)))
        out.append(_window(plan, ptr.value, (int(plan.level_elements[l]),), f"<f{item}"))
    return out


def _rb_windows(plan):
    """per level the GroupedBP recording planes in the plan's storage"""
    out = []
    for l in range(plan.L + 1):
        ptr, n = C.c_void_p(), C.c_uint64()
        capi.check(capi.lib().prodm_mdr_level_rb(plan.h, l, C.byref(ptr), C.byref(n)))
        out.append(_window(plan, ptr.value, (int(n.value),), "|u1"))
    return out


def prepare(case, seed):
    kind, dtype, nb, L = case["kind"], case["dtype"], case["nb"], case["L"]
    dims, enc = _dims(case), _ENC[case["encoder"]]
    st = {"case": case, "kind": kind, "dims": dims, "L": L, "nb": nb}
    if kind in ("step", "streams"):
        hier = bool(case.get("hier"))
        st["x"] = _field(dims, dtype, seed)
        st["plan"] = plan = mdr.Plan(dims, L, nb, _DT[dtype], enc, capi.HIERARCHICAL if hier else capi.ORTHOGONAL)
        st["k"] = _planes_read(L, nb, case.get("full", kind == "streams"))
        if kind == "step":
            if enc == capi.NEGABINARY:
                st["held"] = {"planes": _plane_windows(plan)}
            else:
                st["held"] = {"coefficients": _level_windows(plan)}
                if enc == capi.GROUPED:
                    st["held"]["rb"] = _rb_windows(plan)
            if case["graph"]:
                st["stream"], st["out"] = torch.cuda.Stream(), torch.empty_like(st["x"])
        else:
            plan.refactor(st["x"])
            st["sink"] = mdr.Plan(dims, L, nb, _DT[dtype], enc)
    elif kind == "batch":
        fields = [(_field(d, dtype, seed * 64 + i), d, L) for i, d in enumerate(_batch_shapes(case))]
        st["batch"] = b = batched.Batch(fields, nb, _DT[dtype], enc)
        st["held"] = [_plane_windows(b.plan(f)) for f in range(len(b))]
    elif kind in ("transform", "composed"):
        st["x"] = _field(dims, dtype, seed)
        if kind == "composed":
            st["ld"], _, _ = mdr.level_geometry(dims, L)
    elif kind == "gradient":
        n = math.prod(dims)
        st["x"] = _coefficients(n, dtype, seed).requires_grad_()
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed + 1)
        st["g"] = torch.randn(n, dtype=_DT[dtype], device="cuda", generator=gen)
    else:
        st["x"] = x = _coefficients(dims[0], dtype, seed)
        st["max"] = float(x.abs().max())
        st["exp"] = math.frexp(st["max"])[1]
        if kind == "codec" and enc == capi.PERBIT:
            # the C ABI's caller keeps the buffers
            n, lib, dt = dims[0], capi.lib(), capi.F32 if dtype == "f32" else capi.F64
            st["words"] = int(lib.prodm_perbit_stream_words(n))
            st["streams"] = torch.zeros((nb, st["words"]), dtype=torch.int64, device="cuda")
            st["sizes"] = torch.zeros(nb, dtype=torch.int32, device="cuda")
            st["ws"] = torch.empty(int(lib.prodm_perbit_workspace_bytes(n, nb, dt)), dtype=torch.uint8, device="cuda")
    return st


# ---- one pass -------------------------------------------------------------
def _run_step(st):
    plan = st["plan"]
    if "stream" in st:
        here = torch.cuda.current_stream()
        st["stream"].wait_stream(here)
        with torch.cuda.stream(st["stream"]):
            plan.refactor_graph(st["x"])
            plan.retrieve_graph(st["k"], st["out"])
        here.wait_stream(st["stream"])
        return dict(st["held"], field=st["out"])
    plan.refactor(st["x"])
    return dict(st["held"], field=plan.retrieve(st["k"]))


def _run_composed(st):
    """ComposedRefactor's loop over the components, then ComposedReconstructor's"""
    x, dims, L, nb, ld = st["x"], st["dims"], st["L"], st["nb"], st["ld"]
    coef = mdr.decompose(x, dims, L)
    back = torch.empty_like(x)
    planes = []
    for l in range(L + 1):
        coarse = ld[l - 1] if l else [0] * len(dims)
        buf = mdr.interleave(coef, dims, ld[l], coarse)
        e = math.frexp(mdr.maxabs(buf))[1]
        p = mdr.negabinary_encode(buf, e, nb)
        planes.append(p)
        mdr.reposition(mdr.negabinary_decode(list(p), buf.numel(), e, 0, nb, x.dtype), back, dims, ld[l], coarse)
    return {"planes": planes, "field": mdr.recompose(back, dims, L)}


def _run_streams(st):
    """every plane's bytes to the host, into another plan, and the field from there"""
    a, b, L, nb = st["plan"], st["sink"], st["L"], st["nb"]
    got = [[a.plane_stream(l, p) for p in range(nb)] for l in range(L + 1)]
    for l in range(L + 1):
        b.set_level_max(l, a.level_info(l)[0])
        for p in range(nb):
            b.load_plane_stream(l, p, got[l][p])
    return {"streams": [np.frombuffer(b"".join(level), np.uint8) for level in got], "field": b.retrieve(st["k"])}


def _run_codec(st):
    x, nb, e = st["x"], st["nb"], st["exp"]
    enc = st["case"]["encoder"]
    if enc == "perbit":
        fn = capi.lib().prodm_perbit_encode_f32 if x.dtype == torch.float32 else capi.lib().prodm_perbit_encode_f64
        capi.check(fn(x.data_ptr(), x.numel(), e, nb, 0, st["streams"].data_ptr(), st["words"], st["sizes"].data_ptr(),
                      st["ws"].data_ptr(), st["ws"].numel(), torch.cuda.current_stream().cuda_stream))
        return {"streams": st["streams"], "sizes": st["sizes"]}
    if enc == "grouped":
        rb, planes, words = mdr.grouped_encode(x, e, nb)
        return {"rb": rb, "planes": planes, "words": words}
    planes = mdr.negabinary_encode(x, e, nb)
    k = nb - nb // 4
    return {"planes": planes, "field": mdr.negabinary_decode(list(planes), x.numel(), e, 0, k, x.dtype)}


def run(st):
    kind = st["kind"]
    if kind == "step":
        return _run_step(st)
    if kind == "batch":
        st["batch"].refactor()
        return st["held"]
    if kind == "transform":
        c = mdr.decompose(st["x"], st["dims"], st["L"], hierarchical=st["case"]["hier"])
        return {"coefficients": c, "field": mdr.recompose(c, st["dims"], st["L"], hierarchical=st["case"]["hier"])}
    if kind == "gradient":
        u = autograd.recompose(st["x"], st["dims"], st["L"])
        return {"field": u.detach(), "grad": torch.autograd.grad(u, st["x"], st["g"])[0]}
    if kind == "composed":
        return _run_composed(st)
    if kind == "streams":
        return _run_streams(st)
    if kind == "tables":
        return {"squared": mdr.collect_squared(st["x"], st["nb"], st["max"]),
                "encoder": mdr.level_errors(st["x"], st["exp"], st["nb"])}
    return _run_codec(st)


# ---- what a pass cannot do without ------------------------------------------
def work(case):
    s = 4 if case["dtype"] == "f32" else 8
    nb, L, kind = case["nb"], case["L"], case["kind"]
    if kind == "batch":
        n = sum(math.prod(d) for d in _batch_shapes(case))
        return {"bytes": 2 * s * n, "flops": 40 * n}
    dims = _dims(case)
    n = math.prod(dims)
    if kind == "tables":
        return {"bytes": 2 * s * n, "flops": 4 * (nb + 1) * n}
    if kind == "codec":
        out = nb * n // 8
        # PerBit also stores a sign per element; NegaBinary decodes three quarters of the planes
        more = {"perbit": n // 8, "grouped": n // 8, "negabinary": 3 * out // 4 + s * n}[case["encoder"]]
        return {"bytes": s * n + out + more, "flops": 4 * n}
    if kind == "transform":
        return {"bytes": 4 * s * n, "flops": 80 * n}
    if kind == "gradient":
        return {"bytes": 4 * s * n, "flops": 80 * n}
    if kind == "composed":
        return {"bytes": 2 * s * n + 2 * nb * n // 8, "flops": 80 * n}
    if kind == "streams":
        return {"bytes": 3 * nb * n // 8 + s * n, "flops": 40 * n}
    ld = [[d if d == 1 else ((d - 1) >> (L - l)) + 1 for d in dims] for l in range(L + 1)]
    pts = [math.prod(d) for d in ld]
    read = sum(k * (p - q) // 8 for k, p, q in zip(_planes_read(L, nb, case["full"]), pts, [0] + pts))
    return {"bytes": 2 * s * n + nb * n // 8 + read, "flops": 80 * n}


# ---- the same in 64 bits ----------------------------------------------------
def _project(n):
    """Q = Mc^-1 P^T M along one dim: the coarse part of the L2 projection (c x n)"""
    c = (n >> 1) + 1
    P = torch.zeros(n, c, dtype=torch.float64, device="cuda")
    i = torch.arange(n, device="cuda")
    P[i, i // 2] += 0.5
    P[i, (i + 1) // 2] += 0.5
    M = torch.zeros(n, n, dtype=torch.float64, device="cuda")
    M[i, i] = 2.0
    M[0, 0] = M[-1, -1] = 1.0
    M[i[:-1], i[1:]] = M[i[1:], i[:-1]] = 0.5
    R = P.T @ M
    return torch.linalg.solve(R @ P, R), P


def _along(A, u, d):
    """A applied along dim d"""
    v = u.movedim(d, 0)
    w = A @ v.reshape(v.shape[0], -1)
    return w.reshape([A.shape[0]] + list(v.shape[1:])).movedim(0, d)


def _order(n):
    """natural indices in the decomposed layout's order: even nodes, then odd ones"""
    return torch.cat([torch.arange(0, n, 2), torch.arange(1, n, 2)]).cuda()


def _decompose64(u, L, hier):
    out = u.clone()
    for _ in range(L):
        n = list(u.shape)
        ops = [_project(k) for k in n]
        even = u[tuple(slice(None, None, 2) for _ in n)]
        W, z = even, None
        for d, (_, P) in enumerate(ops):
            W = _along(P, W, d)
        W = u - W
        if not hier:
            z = W
            for d, (Q, _) in enumerate(ops):
                z = _along(Q, z, d)
        box = W
        for d, k in enumerate(n):
            box = box.index_select(d, _order(k))
        out[tuple(slice(0, k) for k in n)] = box
        u = even.clone() if hier else even + z
    out[tuple(slice(0, k) for k in u.shape)] = u
    return out


def _recompose64(c, L):
    dims = list(c.shape)
    ld = [[((d - 1) >> (L - l)) + 1 for d in dims] for l in range(L + 1)]
    u = c[tuple(slice(0, k) for k in ld[0])]
    for l in range(1, L + 1):
        n, low = ld[l], tuple(slice(0, k) for k in ld[l - 1])
        keep = torch.ones(n, dtype=torch.float64, device="cuda")
        keep[low] = 0
        W = c[tuple(slice(0, k) for k in n)] * keep
        for d, k in enumerate(n):
            W = W.index_select(d, torch.argsort(_order(k)))
        ops = [_project(k) for k in n]
        z = W
        for d, (Q, _) in enumerate(ops):
            z = _along(Q, z, d)
        u = u - z
        for d, (_, P) in enumerate(ops):
            u = _along(P, u, d)
        u = u + W
    return u


def _tables64(x, nb, exp):
    x = x.double()
    squared, encoder = [], []
    A, low32 = 0xAAAAAAAA, 0xFFFFFFFF
    s = torch.ldexp(x, torch.tensor(nb - exp - 2, device="cuda"))
    q = s.trunc().to(torch.int64)
    digits = ((q + A) ^ A) & low32
    for k in range(nb + 1):
        t = torch.ldexp(x, torch.tensor(k - exp, device="cuda"))
        d = (t - t.trunc()) * 2.0 ** (exp - k)
        squared.append(float((d * d).sum()))
        v = (((digits & ((1 << (nb - k)) - 1)) ^ A) - A) & low32
        v = torch.where(v >= 1 << 31, v - (1 << 32), v)
        d = v.double() + (s - q.double())
        encoder.append(float((d * d).sum()) * 4.0 ** (exp + 2 - nb))
    return {"squared": np.array(squared), "encoder": np.array(encoder)}


def exact(case, seed):
    kind, L, dims = case["kind"], case["L"], _dims(case)
    if kind in ("step", "streams", "composed"):
        # a retrieval gives the field back, up to the planes that it left out
        return {"field": _field(dims, case["dtype"], seed).double()}
    if kind == "transform":
        u = _field(dims, case["dtype"], seed).double()
        return {"coefficients": _decompose64(u.view(dims), L, case["hier"]).reshape(-1), "field": u}
    if kind == "gradient":
        c = _coefficients(math.prod(dims), case["dtype"], seed).double().requires_grad_()
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed + 1)
        g = torch.randn(c.numel(), dtype=_DT[case["dtype"]], device="cuda", generator=gen).double()
        u = _recompose64(c.view(dims), L).reshape(-1)
        return {"field": u.detach(), "grad": torch.autograd.grad(u, c, g)[0]}
    if kind == "tables":
        x = _coefficients(dims[0], case["dtype"], seed)
        return _tables64(x, case["nb"], math.frexp(float(x.abs().max()))[1])
    if kind == "codec" and case["encoder"] == "negabinary":
        return {"field": _coefficients(dims[0], case["dtype"], seed).double()}
    return None
