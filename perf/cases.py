"""The work that users of this framework have it do, as cases to time and to compare.

A case is one call chain through the public modules: a tensor-product convolution
over an atomistic neighbour graph (``TensorProductConv``), a row-wise product
(``TensorProduct``), or the graph tables a new batch needs
(``TensorProductConv.create_graph``).  Sizes are those of the benchmark and the
tests, or generic ones around them.

Fields of a case: ``kind`` conv | rows | graph; ``mode`` the connection (uvu, uuu,
uvw); ``layout`` full (every path up to ``lmax``) or dot (one 1o x 1o -> 0e path);
``channels``; ``dtype``; ``order`` 0 forward, 1 forward and first derivatives, 2 also
the derivatives of the edge-attribute gradient (energy -> force -> loss training);
``env`` per-edge envelope; ``l0`` per-edge scalar features; ``shared`` one weight row
for every row; ``atoms`` and ``cutoff`` (or ``degree``) the graph; ``rows``.
"""

from __future__ import annotations

import math
from functools import lru_cache

import torch

DENSITY = 0.1  # atoms per cubic Angstrom, as in the benchmark's graphs
DTYPES = {"f32": torch.float32, "f64": torch.float64}


def _case(name, **kw):
    base = dict(kind="conv", mode="uvu", layout="full", lmax=3, channels=64, dtype="f32", order=1,
                env=False, l0=False, shared=False, atoms=0, cutoff=5.0, degree=0, rows=0)
    base.update(kw)
    return dict(name=name, **base) if name else base


def listed():
    return [
        # The smallest call: one forward of a single-path layer on a small fixed-degree
        # graph, as in inference on one molecule. Bound by latency and launches.
        _case("uvu_dot_fwd", layout="dot", lmax=1, channels=32, order=0, atoms=1000, degree=16),
        # The headline layer: one interaction layer's training step on 20,000 atoms.
        _case("uvu_l3_c128_train", channels=128, atoms=20000),
        # The same layer in double precision, as in geometry optimisation and phonons.
        _case("uvu_l3_c128_f64_train", channels=128, dtype="f64", atoms=10000),
        # Force training: energy, forces and the loss's derivatives through the forces.
        _case("uvu_l3_c64_force", channels=64, order=2, atoms=10000),
        # A narrow layer with a cutoff envelope on a small system: the step of a
        # molecular-dynamics run or of a batch of small molecules.
        _case("uvu_l2_c32_env_step", lmax=2, channels=32, env=True, atoms=1000),
        # A ragged channel count, with the per-edge scalar features, evaluated only.
        _case("uvu_l2_c96_l0_fwd", lmax=2, channels=96, order=0, l0=True, atoms=3001, cutoff=4.5),
        # Channel-wise products of node and edge features (per-edge weights), training.
        _case("uuu_l3_c64_train", mode="uuu", atoms=2083),
        # Fully connected convolution with shared weights, training.
        _case("uvw_l3_c64_train", mode="uvw", shared=True, atoms=2083),
        # Fully connected row-wise product with shared weights (node update), training.
        _case("uvw_rows_c64_train", kind="rows", mode="uvw", lmax=2, shared=True, rows=200000),
        # The same product, narrower, in double precision on a smaller batch.
        _case("uvw_rows_c32_f64_train", kind="rows", mode="uvw", lmax=2, channels=32, dtype="f64", shared=True,
              rows=20011),
        # Row-wise product with one shared weight per path and channel, training.
        _case("uvu_rows_c64_train", kind="rows", mode="uvu", lmax=2, shared=True, rows=50000),
        # Graph tables of a new batch: paid on every step whose neighbours change.
        _case("graph_20k", kind="graph", atoms=20000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["uvu", "force", "uuu", "uvw", "uvw_rows", "uvu_rows", "graph"], [6, 2, 2, 2, 3, 2, 1])[0]
    cutoff = round(rng.uniform(3.5, 6.0), 2)
    lmax = rng.choice([1, 2, 2, 3])
    dtype = rng.choices(["f32", "f64"], [3, 1])[0]
    if kind == "graph":
        return _case("", kind="graph", atoms=_log_int(rng, 100, 20000), cutoff=cutoff)
    if kind == "uvw_rows":
        return _case("", kind="rows", mode="uvw", lmax=rng.choice([1, 2]), channels=rng.choice([16, 24, 32, 48, 64]),
                     dtype=dtype, shared=True, rows=_log_int(rng, 500, 100000 if dtype == "f32" else 30000))
    if kind == "uvu_rows":
        return _case("", kind="rows", mode="uvu", lmax=rng.choice([1, 2]), channels=rng.choice([16, 32, 50, 64, 128]),
                     dtype=dtype, shared=rng.random() < 0.7, rows=_log_int(rng, 500, 60000))
    if kind in ("uuu", "uvw"):
        return _case("", mode=kind, lmax=lmax, channels=rng.choice([16, 24, 32, 48, 64]), dtype="f32",
                     shared=kind == "uvw", order=rng.choice([0, 1, 1]), atoms=_log_int(rng, 100, 2083), cutoff=cutoff)
    case = _case("", lmax=lmax, channels=rng.choice([8, 16, 24, 32, 40, 48, 64, 80, 96, 128]), dtype=dtype,
                 order=2 if kind == "force" else rng.choice([0, 1, 1]), cutoff=cutoff,
                 atoms=_log_int(rng, 100, 20000))
    case["env"] = case["order"] < 2 and rng.random() < 0.3
    case["l0"] = case["order"] == 0 and rng.random() < 0.3
    most = 9e9  # bytes of per-edge weights (half of the largest listed case)
    wide = _edges(case) * _layout(case)["wnum"] * (8 if dtype == "f64" else 4)
    if wide > most:
        case["atoms"] = int(case["atoms"] * most / wide)
    return case


# ---------------------------------------------------------------------------
# Layouts: irreps and paths of a case (e3nn's conventions)
# ---------------------------------------------------------------------------

def _name(mul, l, p):
    return f"{mul}x{l}{'e' if p > 0 else 'o'}"


def _layout(case):
    key = tuple(case[k] for k in ("kind", "mode", "layout", "lmax", "channels"))
    return _layout_of(*key)


@lru_cache(maxsize=None)
def _layout_of(kind, mode, layout, lmax, channels):
    """Irreps strings, instructions and, per path, offsets and its normalised coefficient."""
    degrees = [1] if layout == "dot" else list(range(lmax + 1))
    parity = lambda l: 1 if l % 2 == 0 else -1  # noqa: E731
    in1 = [(channels, l, parity(l)) for l in degrees]
    in2 = [(channels if mode == "uuu" else 1, l, parity(l)) for l in degrees]
    outs, instructions = [], []
    if mode == "uvu":  # every path has an output block of its own
        for i, (_, l1, p1) in enumerate(in1):
            for j, (_, l2, p2) in enumerate(in2):
                for l3 in range(abs(l1 - l2), l1 + l2 + 1):
                    if l3 <= lmax and (layout == "full" or l3 == 0):
                        instructions.append((i, j, len(outs), mode, True))
                        outs.append((channels, l3, p1 * p2))
    else:  # paths are summed into the input's irreps
        outs = list(in1)
        instructions = [(i, j, k, mode, True) for i, a in enumerate(in1) for j, b in enumerate(in2)
                        for k, c in enumerate(outs)
                        if abs(a[1] - b[1]) <= c[1] <= a[1] + b[1] and a[2] * b[2] == c[2]]
    starts = lambda irreps: [sum(m * (2 * l + 1) for m, l, _ in irreps[:n]) for n in range(len(irreps) + 1)]  # noqa: E731
    s1, s2, s3 = starts(in1), starts(in2), starts(outs)
    paths, wnum = [], 0
    for i, j, k, _, _ in instructions:
        fan = sum({"uvu": 1, "uuu": 1, "uvw": channels}[mode] for ins in instructions if ins[2] == k)
        l1, l2, l3 = in1[i][1], in2[j][1], outs[k][1]
        paths.append(dict(l1=l1, l2=l2, l3=l3, x=s1[i], y=s2[j], o=s3[k], w=wnum,
                          c=math.sqrt((2 * l3 + 1) / fan)))
        wnum += channels * channels if mode == "uvw" else channels
    text = lambda irreps: "+".join(_name(*ir) for ir in irreps)  # noqa: E731
    return dict(in1=text(in1), in2=text(in2), out=text(outs), instructions=instructions, paths=paths,
                wnum=wnum, d1=s1[-1], d2=s2[-1], d3=s3[-1])


def _edges(case):
    """Number of edges: the fixed degree, or the expected neighbours at this density."""
    if case["degree"]:
        return case["atoms"] * case["degree"]
    around = min(DENSITY * 4 / 3 * math.pi * case["cutoff"] ** 3, case["atoms"] - 1)
    return int(case["atoms"] * around)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

_modules = {}


def _module(case):
    """The layer: a program builds it once and keeps it."""
    from lunaequivariance_amd import TensorProduct, TensorProductConv

    key = tuple(case[k] for k in ("kind", "mode", "layout", "lmax", "channels", "dtype", "shared"))
    if key not in _modules:
        if len(_modules) > 40:
            _modules.clear()
        lay = _layout(case)
        cls = TensorProductConv if case["kind"] == "conv" else TensorProduct
        _modules[key] = cls(lay["in1"], lay["in2"], lay["out"], lay["instructions"], shared_weights=case["shared"],
                            internal_weights=False, dtype=DTYPES[case["dtype"]]).to("cuda")
    return _modules[key]


def _neighbours(case, seed):
    """(src, dst, unit vectors) on the GPU, sorted by dst: the radius graph of random atoms
    in a periodic cube, or random sources at a fixed degree."""
    gen = torch.Generator(device="cuda").manual_seed(seed * 7919 + 11)
    n = case["atoms"]
    if case["degree"]:
        dst = torch.arange(n, device="cuda").repeat_interleave(case["degree"])
        src = torch.randint(0, n, dst.shape, device="cuda", generator=gen)
        vec = torch.randn(len(dst), 3, device="cuda", dtype=torch.float64, generator=gen)
        return src, dst, vec / vec.norm(dim=1, keepdim=True)
    box = (n / DENSITY) ** (1 / 3)
    pos = torch.rand(n, 3, device="cuda", dtype=torch.float64, generator=gen) * box
    # Exactly the expected number of edges, so that sizes depend on the case alone: the
    # nearest pairs, i.e. the cutoff moves a little from one set of positions to another.
    edges, radius = _edges(case), case["cutoff"]
    while True:
        radius *= 1.05
        found = []
        for lo in range(0, n, 2048):
            delta = pos[None] - pos[lo:lo + 2048, None]
            delta -= box * torch.round(delta / box)
            dist2 = (delta * delta).sum(-1)
            dist2[torch.arange(dist2.shape[0]), torch.arange(lo, lo + dist2.shape[0])] = math.inf
            dst, src = (dist2 < radius * radius).nonzero(as_tuple=True)
            found.append((src, dst + lo, dist2[dst, src], delta[dst, src]))
        src, dst, dist2, vec = (torch.cat(t) for t in zip(*found))
        if len(src) >= edges:
            break
    keep = torch.sort(dist2, stable=True).indices[:edges].sort().values
    src, dst, vec = src[keep], dst[keep], vec[keep]
    return src, dst, vec / vec.norm(dim=1, keepdim=True)


def _harmonics(lmax, v):
    """Real spherical harmonics of unit vectors, component normalised, in the (y, z, x) order."""
    x, y, z = v.unbind(1)
    out = [torch.ones_like(x)[:, None], math.sqrt(3) * v]
    if lmax >= 2:
        s = math.sqrt(15)
        out.append(torch.stack([s * x * z, s * x * y, math.sqrt(5) * (y * y - (x * x + z * z) / 2), s * y * z,
                                s / 2 * (z * z - x * x)], 1))
    if lmax >= 3:
        a, b, r = math.sqrt(70) / 4, math.sqrt(105), math.sqrt(42) / 4
        out.append(torch.stack([a * x * (3 * z * z - x * x), b * x * y * z, r * x * (4 * y * y - x * x - z * z),
                                math.sqrt(7) / 2 * y * (2 * y * y - 3 * x * x - 3 * z * z),
                                r * z * (4 * y * y - x * x - z * z), b / 2 * y * (z * z - x * x),
                                a * z * (z * z - 3 * x * x)], 1))
    return torch.cat(out[:lmax + 1], 1)


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, lay = DTYPES[case["dtype"]], _layout(case)
    normal = lambda *shape: torch.randn(*shape, device="cuda", dtype=dtype, generator=gen)  # noqa: E731
    if case["kind"] == "rows":
        nodes = edges = case["rows"]
        s = {}
        vec = torch.randn(edges, 3, device="cuda", dtype=torch.float64, generator=gen)
        vec = vec / vec.norm(dim=1, keepdim=True)
    else:
        src, dst, vec = _neighbours(case, seed)
        nodes, edges = case["atoms"], len(src)
        s = {"src": src, "dst": dst}
        if case["kind"] == "graph":
            return s
    s["x"] = normal(nodes, lay["d1"])
    if case["mode"] == "uuu":
        s["y"] = normal(edges, lay["d2"])
    elif case["layout"] == "dot":
        s["y"] = vec.to(dtype)
    else:
        s["y"] = _harmonics(case["lmax"], vec).to(dtype)
    s["w"] = normal(lay["wnum"]) if case["shared"] else normal(edges, lay["wnum"])
    s["env"] = torch.rand(edges, device="cuda", dtype=dtype, generator=gen) if case["env"] else None
    if case["order"]:
        s["g"] = normal(nodes, lay["d3"])
    if case["order"] == 2:
        s["ry"] = normal(edges, lay["d2"])
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "graph":
        return dict(case=case, **s)
    module = _module(case)
    if case["kind"] == "conv":
        s["graph"] = module.create_graph(s.pop("src"), s.pop("dst"), case["atoms"])
    if case["order"]:
        for name in ("x", "y", "w", "env") + (("g",) if case["order"] == 2 else ()):
            if s[name] is not None:
                s[name].requires_grad_()
    return dict(case=case, module=module, **s)


def run(state):
    case = state["case"]
    if case["kind"] == "graph":
        from lunaequivariance_amd import TensorProductConv

        g = TensorProductConv.create_graph(state["src"], state["dst"], case["atoms"])
        return {"dst_rowptr": g.dst_rowptr, "src_rowptr": g.src_rowptr, "edge_ids_by_src": g.edge_ids_by_src,
                "node_order": g.node_order, "source_node_order": g.source_node_order}
    x, y, w = state["x"], state["y"], state["w"]
    if case["kind"] == "rows":
        out = state["module"](x, y, w)
    else:
        kw = {}
        if case["env"]:
            kw["env"] = state["env"]
        if case["l0"]:
            kw["return_l0_feat"] = True
        out = state["module"](x, y, w, graph=state["graph"], **kw)
    if not case["order"]:
        return {"out": out[0], "l0": out[1]} if case["l0"] else {"out": out}
    args = [x, y, w] + ([state["env"]] if case["env"] else [])
    grads = torch.autograd.grad(out, args, state["g"], create_graph=case["order"] == 2)
    result = dict(zip(("gx", "gy", "gw", "genv"), grads), out=out)
    if case["order"] == 2:
        result.update(zip(("hx", "hw", "hg"), torch.autograd.grad(grads[1], (x, w, state["g"]), state["ry"])))
    return {k: v.detach() for k, v in result.items()}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    b = 8 if case["dtype"] == "f64" else 4
    lay = _layout(case)
    n, e = (case["rows"],) * 2 if case["kind"] == "rows" else (case["atoms"], _edges(case))
    if case["kind"] == "graph":  # 64-bit sources and destinations in, 32-bit tables out
        return {"bytes": 16 * e + 4 * e + 16 * n, "flops": 0}
    x, y, out = n * lay["d1"], e * lay["d2"], n * lay["d3"]
    w = lay["wnum"] if case["shared"] else e * lay["wnum"]
    total = x + y + w + out + (e if case["env"] else 0)
    if case["l0"]:
        total += e * sum(case["channels"] for p in lay["paths"] if p["l3"] == 0)
    if case["order"]:
        total += x + y + w + out + (e if case["env"] else 0)
    if case["order"] == 2:
        total += y + x + w + out
    index = 0 if case["kind"] == "rows" else (8 * e + 8 * n if case["order"] else 4 * e + 4 * n)
    c, terms = case["channels"], sum(int((_cg(p["l1"], p["l2"], p["l3"]).abs() > 1e-9).sum()) for p in lay["paths"])
    comps = sum(2 * p["l3"] + 1 for p in lay["paths"])
    per = {0: 1, 1: 3, 2: 6}[case["order"]]
    flops = e * c * (3 * terms + 2 * comps)
    if case["mode"] == "uvw":  # shared weights: one contraction per node or row
        flops += n * 2 * c * c * comps
    return {"bytes": total * b + index, "flops": per * flops}


def tolerance(case):
    if case["kind"] == "graph":
        return "exact"
    # About four times the largest error measured against exact(): 5.8e-7 (f32) and 9.7e-15
    # (f64), both of a weight gradient summed over the rows.
    return {"rel": 4e-14, "max": 4e-12} if case["dtype"] == "f64" else {"rel": 2.5e-6, "max": 1e-4}


# ---------------------------------------------------------------------------
# The same results from the definition, in 64 bits
# ---------------------------------------------------------------------------

@lru_cache(maxsize=None)
def _cg(l1, l2, l3):
    """Real coupling coefficients [2 l1 + 1, 2 l2 + 1, 2 l3 + 1] of unit norm: Racah's formula
    for <l1 m1 l2 m2 | l3 m3>, taken to the real harmonics whose phase is (-i)^l."""
    f = math.factorial
    complex_cg = torch.zeros(2 * l1 + 1, 2 * l2 + 1, 2 * l3 + 1, dtype=torch.complex128)
    lead = (2 * l3 + 1) * f(l3 + l1 - l2) * f(l3 - l1 + l2) * f(l1 + l2 - l3) / f(l1 + l2 + l3 + 1)
    for m1 in range(-l1, l1 + 1):
        for m2 in range(-l2, l2 + 1):
            m3 = m1 + m2
            if abs(m3) > l3:
                continue
            total = 0.0
            for k in range(l1 + l2 - l3 + 1):
                below = (l1 + l2 - l3 - k, l1 - m1 - k, l2 + m2 - k, l3 - l2 + m1 + k, l3 - l1 - m2 + k)
                if min(below) >= 0:
                    total += (-1) ** k / math.prod(f(v) for v in below) / f(k)
            scale = math.prod(f(l + m) * f(l - m) for l, m in ((l1, m1), (l2, m2), (l3, m3)))
            complex_cg[l1 + m1, l2 + m2, l3 + m3] = math.sqrt(lead * scale) * total

    def basis(l):
        q = torch.zeros(2 * l + 1, 2 * l + 1, dtype=torch.complex128)  # complex m from real m'
        q[l, l] = 1
        for m in range(1, l + 1):
            sign = (-1) ** m
            q[l - m, l + m], q[l - m, l - m] = 1 / math.sqrt(2), -1j / math.sqrt(2)
            q[l + m, l + m], q[l + m, l - m] = sign / math.sqrt(2), sign * 1j / math.sqrt(2)
        return (-1j) ** l * q

    real = torch.einsum("abc,ai,bj,ck->ijk", complex_cg, basis(l1), basis(l2), basis(l3).conj()).real
    return real / real.norm()


def _messages(case, x, y, w):
    """Per-edge (or per-row) products, [edges, d3]; for uvw the aggregate blocks before the weights."""
    lay, ch, e = _layout(case), case["channels"], x.shape[0]
    parts = {}
    scalars = []
    for n, p in enumerate(lay["paths"]):
        d1, d2, d3 = 2 * p["l1"] + 1, 2 * p["l2"] + 1, 2 * p["l3"] + 1
        cg = _cg(p["l1"], p["l2"], p["l3"]).to(x.device) * p["c"]
        xp = x[:, p["x"]:p["x"] + ch * d1].reshape(e, ch, d1)
        if case["mode"] == "uuu":
            z = (y[:, p["y"]:p["y"] + ch * d2].reshape(-1, d2) @ cg.permute(1, 0, 2).reshape(d2, -1))
            m = (xp[..., None] * z.reshape(e, ch, d1, d3)).sum(2)
        else:
            z = (y[:, p["y"]:p["y"] + d2] @ cg.permute(1, 0, 2).reshape(d2, -1)).reshape(e, d1, d3)
            m = torch.bmm(xp, z)
        if case["mode"] != "uvw":
            m = m * w[..., p["w"]:p["w"] + ch, None]
            if p["l3"] == 0:
                scalars.append(m[..., 0])
            parts[p["o"]] = parts.get(p["o"], 0) + m.reshape(e, -1)
        else:
            parts[n] = m
    if case["mode"] == "uvw":
        return parts
    return torch.cat([parts[o] for o in sorted(parts)], 1), scalars


def _contract(case, parts, w):
    ch, out = case["channels"], {}
    for n, p in enumerate(_layout(case)["paths"]):
        m = torch.einsum("ncd,cw->nwd", parts[n], w[p["w"]:p["w"] + ch * ch].reshape(ch, ch))
        out[p["o"]] = out.get(p["o"], 0) + m.reshape(m.shape[0], -1)
    return torch.cat([out[o] for o in sorted(out)], 1)


def exact(case, seed):
    if case["kind"] == "graph":
        return None
    s = _inputs(case, seed)
    up = lambda t: None if t is None else t.double()  # noqa: E731
    x, w, env = up(s["x"]), s["w"], s["env"]
    nodes, lay, order = x.shape[0], _layout(case), case["order"]
    rows = case["kind"] == "rows"
    if case["shared"]:
        w = w.double()
    result = {}

    def into(name, value, lo=0, hi=None):
        """Adds node or shared results; stores the rows [lo, hi) of per-edge ones."""
        if hi is None:
            result[name] = result[name] + value if name in result else value
        else:
            if name not in result:
                result[name] = torch.empty((edges,) + value.shape[1:], device=value.device, dtype=torch.float64)
            result[name][lo:hi] = value

    edges = s["y"].shape[0]
    if case["mode"] == "uvw" and not rows:
        step = edges  # the weights come after the sum over edges
    else:
        step = max(256, int(2e9 / (8 * 12 * (lay["d1"] + lay["d3"]) + 16 * lay["wnum"] * (not case["shared"]))))
    for lo in range(0, edges, step):
        hi = min(lo + step, edges)
        # x is taken by rows where every row is its own node, else whole.
        xc = x[lo:hi] if rows else x
        leaves = {"x": xc.detach(), "y": s["y"][lo:hi].double(), "w": w if case["shared"] else w[lo:hi].double()}
        if env is not None:
            leaves["env"] = env[lo:hi].double()
        if order:
            gc = s["g"][lo:hi].double() if rows else s["g"].double()
            leaves = {k: v.detach().requires_grad_() for k, v in leaves.items()}
            gc.requires_grad_(order == 2)
        at = leaves["x"] if rows else leaves["x"][s["src"][lo:hi]]
        if case["mode"] == "uvw":
            parts = _messages(case, at, leaves["y"], None)
            if not rows:
                parts = {n: m.new_zeros(nodes, *m.shape[1:]).index_add(0, s["dst"], m) for n, m in parts.items()}
            out = _contract(case, parts, leaves["w"])
        else:
            m, scalars = _messages(case, at, leaves["y"], leaves["w"])
            if case["l0"]:
                into("l0", torch.cat(scalars, 1), lo, hi)
            if env is not None:
                m = m * leaves["env"][:, None]
            out = m if rows else m.new_zeros(nodes, lay["d3"]).index_add(0, s["dst"][lo:hi], m)
        per = (lo, hi)
        into("out", out.detach(), *(per if rows else ()))
        if order:
            grads = torch.autograd.grad(out, list(leaves.values()), gc, create_graph=order == 2)
            named = dict(zip(["g" + k for k in leaves], grads))
            if order == 2:
                wanted = {"hx": leaves["x"], "hw": leaves["w"], "hg": gc}
                named.update(zip(wanted, torch.autograd.grad(named["gy"], list(wanted.values()),
                                                             s["ry"][lo:hi].double())))
            for name, value in named.items():
                whole = {"x": not rows, "g": not rows, "w": case["shared"]}.get(name[1:], False)
                into(name, value.detach(), *(() if whole else per))
    return result
