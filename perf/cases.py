"""Cases of use of the framework, for measuring it: what a program does with it,
from a small cell whose cost is latency to the largest systems of the benchmark.

Four kinds of calls, each through the Python binding:

  md      a short NVE segment of a device-resident system: set_positions and
          set_velocities (the start of a trajectory, e.g. one replica of many),
          md_run with its energy history, and get;
  static  one evaluation driven from outside (relaxation, a path-integral
          driver): set_positions and compute, which returns every result;
  list    the Pair::compute drop-in over a LAMMPS full neighbor list with ghost
          atoms: either every call brings its list (the call after a neighbor
          build), or the list's serial is unchanged (the calls between two
          builds, which send positions only);
  serve   the request loop over periodic structures of mixed sizes: one request
          at a time, or a burst of requests.

Models are random-init with the shapes of the repository's tests, golden files
and benchmark.  Crystals are jittered lattices (0.05 to 0.1 A), as there.

The entry points return 64-bit arrays whatever the arithmetic behind the
values.  Here every value comes back in the type of its arithmetic: 32 bits,
and where the model's network runs on 8-bit significands (bf16, fp8), bfloat16
for what the network's output makes (energies, forces, virials); positions,
velocities and kinetic energies stay at 32 bits there too.
"""
import atexit
import math
import os
import shutil
import sys
import tempfile

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "lammps-tensormd_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from tensormd_amd import NeighborList, TensorMD  # noqa: E402
from tensormd_amd import workloads as W  # noqa: E402

SKIN = 1.0   # A, of lists and device systems
DT = 0.001   # ps

# The model shapes: the 1-element and 4-element networks of the benchmark
# configurations (tanh), the wider 4-element one of its 8-bit experiment, the
# 2-element squareplus network with skips of the tests, and the shape of the
# 1-element production file (64 filters, 128-wide squareplus network).
MODELS = {
    "fcc1": dict(symbols=["Cu"], masses=[63.546], rmax=6.0, num_filters=16,
                 layer_sizes=[128, 64, 1], actfn="tanh", seed=11, radial_scale=0.2),
    "bcc4": dict(symbols=["Mo", "Nb", "Ta", "W"], masses=[95.95, 92.906, 180.95, 183.84],
                 rmax=6.5, num_filters=24, layer_sizes=[256, 128, 64, 1], actfn="tanh",
                 seed=12, radial_scale=0.2),
    "bcc4w": dict(symbols=["Mo", "Nb", "Ta", "W"], masses=[95.95, 92.906, 180.95, 183.84],
                  rmax=6.5, num_filters=24, layer_sizes=[256, 256, 128, 1], actfn="tanh",
                  seed=5, radial_scale=0.2),
    "fcc2": dict(symbols=["Al", "Ni"], masses=[26.98, 58.69], rmax=5.5, num_filters=32,
                 layer_sizes=[64, 64, 64, 1], actfn="squareplus", use_resnet_dt=True, seed=13,
                 radial_scale=0.2),
    "bcc1k64": dict(symbols=["W"], masses=[183.84], rmax=6.0, num_filters=64,
                    layer_sizes=[128, 128, 128, 128, 1], actfn="squareplus",
                    use_resnet_dt=True, seed=17, radial_scale=0.2),
}
# lattice, constant (A), jitter (A), temperature (K) of each model's crystals
CRYSTAL = {"fcc1": ("fcc", 3.615, 0.05, 300.0), "bcc4": ("bcc", 3.2, 0.08, 600.0),
           "bcc4w": ("bcc", 3.2, 0.08, 600.0), "fcc2": ("fcc", 3.8, 0.06, 300.0),
           "bcc1k64": ("bcc", 3.18, 0.08, 600.0)}


def listed():
    return [
        # the smallest trajectory: launches and latency
        dict(name="md small fp32", kind="md", model="bcc4", mode="fp32", nx=4, ny=4, nz=4, steps=20),
        # the 2,048-atom one-element configuration
        dict(name="md fcc 2k fp32", kind="md", model="fcc1", mode="fp32", nx=8, ny=8, nz=8, steps=20),
        # a mid-size alloy in plain FP32
        dict(name="md bcc 16k fp32", kind="md", model="bcc4", mode="fp32", nx=20, ny=20, nz=20, steps=10),
        # odd sizes, the split-BF16 network
        dict(name="md bcc 38k bf16x3", kind="md", model="bcc4", mode="bf16x3", nx=27, ny=29, nz=25, steps=8),
        # the headline system
        dict(name="md bcc 128k bf16", kind="md", model="bcc4", mode="bf16", nx=40, ny=40, nz=40, steps=10),
        # the wide network's 8-bit experiment, at a size between the two large systems
        dict(name="md bcc 250k fp8", kind="md", model="bcc4w", mode="fp8", nx=50, ny=50, nz=50, steps=4),
        # one relaxation step of a two-element alloy, network with skips
        dict(name="static fcc2 2772 fp32", kind="static", model="fcc2", mode="fp32", nx=11, ny=9, nz=7),
        # one evaluation of the one-element production shape
        dict(name="static k64 11k bf16", kind="static", model="bcc1k64", mode="bf16", nx=18, ny=18, nz=17),
        # a LAMMPS step right after a neighbor build, per-atom energies and virials asked for
        dict(name="list fcc 2k fp32", kind="list", model="fcc1", mode="fp32", nx=8, ny=8, nz=8,
             reuse=False, vatom=True),
        # the LAMMPS steps between two neighbor builds
        dict(name="list reuse 31k bf16", kind="list", model="bcc4", mode="bf16", nx=25, ny=25, nz=25,
             reuse=True, vatom=False),
        # one request at a time: latency of a small structure
        dict(name="serve one fp32", kind="serve", model="bcc4", mode="fp32", count=1, nmin=54, nmax=54),
        # a burst of requests of mixed sizes
        dict(name="serve burst bf16", kind="serve", model="bcc4", mode="bf16", count=192, nmin=16, nmax=4096),
    ]


def _cells(rng, lo, hi, basis):
    """Ragged supercell of about a log-uniform number of atoms in [lo, hi]."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi))) / basis
    side = n ** (1.0 / 3.0)
    out = [max(3, round(side * rng.uniform(0.8, 1.25))) for _ in range(2)]
    out.append(max(3, round(n / (out[0] * out[1]))))
    while out[0] * out[1] * out[2] * basis > hi and max(out) > 3:
        out[out.index(max(out))] -= 1
    return dict(nx=out[0], ny=out[1], nz=out[2])


def draw(rng):
    kind = rng.choice(["md", "md", "md", "static", "list", "serve"])
    if kind == "md":
        model = rng.choice(["bcc4", "bcc4", "fcc1"])
        mode = rng.choice(["fp32", "bf16", "bf16x3"] if model == "bcc4" else ["fp32", "bf16"])
        hi = 24000 if mode == "fp32" else (110000 if mode == "bf16" else 48000)
        return dict(kind=kind, model=model, mode=mode, steps=rng.randint(4, 12),
                    **_cells(rng, 128, hi, 2 if model == "bcc4" else 4))
    if kind == "static":
        model = rng.choice(["fcc2", "bcc1k64", "bcc4w"])
        mode = rng.choice(["fp32", "bf16"]) if model != "bcc4w" else "fp8"
        return dict(kind=kind, model=model, mode=mode,
                    **_cells(rng, 200, 16000, 4 if model == "fcc2" else 2))
    if kind == "list":
        model = rng.choice(["fcc1", "bcc4"])
        return dict(kind=kind, model=model, mode=rng.choice(["fp32", "bf16"]),
                    reuse=rng.random() < 0.6, vatom=rng.random() < 0.3,
                    **_cells(rng, 500, 30000, 4 if model == "fcc1" else 2))
    count = 1 if rng.random() < 0.3 else rng.randint(8, 192)
    nmin = rng.randint(16, 54)
    return dict(kind=kind, model="bcc4", mode=rng.choice(["fp32", "bf16"]), count=count,
                nmin=nmin, nmax=nmin if count == 1 else rng.randint(256, 4096))


# ---------------------------------------------------------------------------
_files = {}


def _model_file(model):
    """The model file of a shape, written once by this process."""
    if model not in _files:
        d = tempfile.mkdtemp(prefix="tmd_cases_")
        atexit.register(shutil.rmtree, d, ignore_errors=True)
        _files[model] = W.write_model(os.path.join(d, model + ".npz"), **MODELS[model])
    return _files[model]


def _structure(case, seed):
    """Positions, types and cell of a case's crystal, and its velocities."""
    m = MODELS[case["model"]]
    lat, a, sigma, temp = CRYSTAL[case["model"]]
    x, types, cell = W.crystal(lat, a, (case["nx"], case["ny"], case["nz"]),
                               nelt=len(m["symbols"]), sigma=sigma, seed=seed)
    mass = np.array(m["masses"])[types - 1]
    return x, types, cell, W.maxwell_boltzmann(mass, temp, seed=seed + 1)


def _requests(case, seed):
    """The case's mix of structures, with occupation and displacements of the seed."""
    rng = np.random.default_rng(seed)
    mix = W.serving_requests(case["count"], seed=case["count"], nmin=case["nmin"],
                             nmax=case["nmax"], sigma=0.08)
    return [(W.wrap(x + rng.normal(0.0, 0.06, size=x.shape), cell),
             rng.integers(1, 5, size=len(x)).astype(np.int32), cell) for x, _, cell in mix]


def _box(cell):
    return np.diagonal(cell).copy()


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _pairs(x, length, cut):
    """Pairs (i, j, image) within `cut` in a box of edges `length`, sorted by
    i: atoms and their images are binned into cells at least `cut` wide, and
    every atom meets the 27 cells around its own.  image indexes the returned
    list of ghost positions and owners (the atoms themselves first)."""
    dev = _device()
    x = torch.as_tensor(x, dtype=torch.float64, device=dev)
    length = torch.as_tensor(length, dtype=torch.float64, device=dev)
    n = x.shape[0]
    reach = [int(math.ceil(cut / float(v))) for v in length]
    pos, owner = [x], [torch.arange(n, device=dev)]
    for a in range(-reach[0], reach[0] + 1):
        for b in range(-reach[1], reach[1] + 1):
            for c in range(-reach[2], reach[2] + 1):
                if a == b == c == 0:
                    continue
                y = x + torch.tensor([a, b, c], dtype=torch.float64, device=dev) * length
                near = ((y > -cut) & (y < length + cut)).all(1).nonzero()[:, 0]
                pos.append(y[near])
                owner.append(near)
    pos, owner = torch.cat(pos), torch.cat(owner)
    nb = torch.floor((length + 2 * cut) / cut).long().clamp(min=1)
    width = (length + 2 * cut) / nb
    cell = torch.minimum(((pos + cut) / width).long().clamp(min=0), nb - 1)
    nb1 = nb + 2  # an empty shell around the cells
    flat = ((cell[:, 0] + 1) * nb1[1] + cell[:, 1] + 1) * nb1[2] + cell[:, 2] + 1
    order = torch.argsort(flat, stable=True)
    count = torch.bincount(flat, minlength=int(nb1.prod()))
    start = torch.cumsum(count, 0) - count
    out_i, out_j = [], []
    for lo in range(0, n, 8192):
        mine = torch.arange(lo, min(n, lo + 8192), device=dev)
        for a in (-1, 0, 1):
            for b in (-1, 0, 1):
                for c in (-1, 0, 1):
                    q = flat[mine] + (a * nb1[1] + b) * nb1[2] + c
                    m = count[q]
                    i = torch.repeat_interleave(mine, m)
                    first = torch.repeat_interleave(start[q] - (torch.cumsum(m, 0) - m), m)
                    j = order[first + torch.arange(i.numel(), device=dev)]
                    d = pos[j] - pos[i]
                    ok = ((d * d).sum(1) <= cut * cut) & (i != j)
                    out_i.append(i[ok])
                    out_j.append(j[ok])
    i, j = torch.cat(out_i), torch.cat(out_j)
    order = torch.argsort(i, stable=True)
    return i[order], j[order], pos, owner


def prepare(case, seed):
    m = MODELS[case["model"]]
    model = TensorMD(_model_file(case["model"]), m["symbols"], case["mode"], 0.001, device=0)
    state = dict(case=case, model=model)
    if case["kind"] == "serve":
        state["requests"] = _requests(case, seed)
        state["arrival"] = np.zeros(case["count"])
        state["server"] = model.serve()
        return state
    x, types, cell, v = _structure(case, seed)
    if case["kind"] in ("md", "static"):
        state.update(x=x, v=v, system=model.system(x, types, cell, skin=SKIN))
        return state
    i, j, pos, owner = _pairs(x, _box(cell), m["rmax"] + SKIN)
    n = len(x)
    state.update(x=pos.cpu().numpy(), types=types[owner.cpu().numpy()],
                 list=NeighborList(n, np.arange(n), torch.bincount(i, minlength=n).cpu().numpy(),
                                   j.cpu().numpy()))
    state["out"] = dict(f=np.zeros((len(pos), 3)), eatom=np.zeros(n),
                        vatom=np.zeros((len(pos), 6)) if case["vatom"] else None, energy=0.0,
                        virial=np.zeros(6))
    return state


def _types(case):
    """Output types: of what the network's output makes, and of the rest."""
    return (torch.bfloat16 if case["mode"] in ("bf16", "fp8") else torch.float32), torch.float32


def _out(a, dtype):
    return None if a is None else torch.as_tensor(a).to(dtype)


def run(state):
    case = state["case"]
    net, rest = _types(case)
    if case["kind"] == "md":
        s = state["system"]
        s.set_positions(state["x"])
        s.set_velocities(state["v"])
        epot, ekin = s.md_run(case["steps"], DT)
        r = s.get()
        return dict(x=_out(r["x"], rest), v=_out(r["v"], rest), f=_out(r["f"], net),
                    eatom=_out(r["eatom"], net), virial=_out(r["virial"], net),
                    epot=_out(epot, net), ekin=_out(ekin, rest))
    if case["kind"] == "static":
        s = state["system"]
        s.set_positions(state["x"])
        r = s.compute()
        return dict(f=_out(r["f"], net), eatom=_out(r["eatom"], net),
                    virial=_out(r["virial"], net), energy=_out(r["energy"], net))
    if case["kind"] == "list":
        r = state["model"].compute_list_ptrs(state["list"], state["x"], state["types"],
                                             serial=1 if case["reuse"] else None, out=state["out"])
        return dict(f=_out(r["f"], net), eatom=_out(r["eatom"], net), vatom=_out(r["vatom"], net),
                    virial=_out(r["virial"], net), energy=_out(r["energy"], net))
    if case["count"] == 1:
        res = [state["server"].wait(state["server"].submit(*state["requests"][0]))]
        f = [res[0]["f"]]
    else:
        res, f = state["server"].replay(state["requests"], state["arrival"])
    return dict(f=_out(np.concatenate(f), net), virial=_out(np.stack([r["virial"] for r in res]), net),
                energy=_out(np.array([r["energy"] for r in res]), net))


# ---------------------------------------------------------------------------
def _atoms(case):
    """Atoms of one pass and evaluations of each."""
    if case["kind"] == "serve":
        return sum(len(r[0]) for r in _requests(case, 1)), 1
    basis = 2 if CRYSTAL[case["model"]][0] == "bcc" else 4
    return case["nx"] * case["ny"] * case["nz"] * basis, case.get("steps", 0) + 1


def work(case):
    """Per evaluation and atom: the radial functions and the moments of its
    neighbors (16 independent harmonics up to degree 3 per filter), the
    network forward and backward, the chain rule; the list, positions and
    forces, and the descriptor rows and their gradients, which every path
    hands through memory between the per-atom and the per-tile work."""
    m = MODELS[case["model"]]
    lat, a, _, _ = CRYSTAL[case["model"]]
    density = (2 if lat == "bcc" else 4) / a ** 3
    c = 4.0 / 3.0 * math.pi * m["rmax"] ** 3 * density
    k, b = m["num_filters"], len(m["symbols"])
    width = 4 * k * b
    sizes = [width] + m["layer_sizes"]
    mlp = 4 * sum(p * q for p, q in zip(sizes[:-1], sizes[1:]))
    g = 2 if case["mode"] == "bf16" else 4
    atoms, evals = _atoms(case)
    return {"flops": atoms * evals * (mlp + 2 * c * 16 * k * 3 + 19 * c * k),
            "bytes": atoms * evals * (2 * 4 * c + 2 * 32 + 2 * 24 + 2 * (g + 4) * width)}


# ---------------------------------------------------------------------------
# The same results in 64 bits, in plain torch.
def _weights(model, dev):
    with np.load(_model_file(model), allow_pickle=False) as z:
        return {k: torch.as_tensor(z[k], device=dev) for k in z.files}


def _table(model, w, dev):
    """Radial functions at the grid points and the interpolant's coefficients
    per cell: value, slope, and the two second differences (zero in the end
    cells), as the model's table defines them at 0.001 A."""
    dx = 0.001
    n = int(MODELS[model]["rmax"] / dx) + 1
    r = torch.arange(n, dtype=torch.float64, device=dev) * dx
    h = r[:, None]
    last = int(w["fnn::nlayers"]) - 1
    for q in range(last + 1):
        h = h @ w["fnn::weights_0_%d" % q].reshape(h.shape[1], -1)
        if q < last:
            h = torch.nn.functional.softplus(h + w["fnn::biases_0_%d" % q], threshold=1e9)
    y = h * (0.5 + 0.5 * torch.cos(torch.clamp(r / MODELS[model]["rmax"], max=1.0) * math.pi))[:, None]
    s = (y[1:] - y[:-1]) / dx
    c1, c2 = torch.zeros_like(s), torch.zeros_like(s)
    c1[1:] = (s[1:] - s[:-1]) / (2 * dx)
    c2[:-1] = (s[1:] - s[:-1]) / (2 * dx)
    return y, s, c1, c2, dx


def _radial(tab, r):
    y, s, c1, c2, dx = tab
    n = torch.clamp((r.detach() * (1.0 / dx)).long(), max=s.shape[0] - 1)
    live = ((n > 0) & (n < s.shape[0] - 1))[:, None]
    q = (r - n.to(r.dtype) * dx)[:, None]
    p = dx - q
    a, b = c1[n], c2[n]
    num = (b * p).abs()
    den = num + (a * q).abs()
    wgt = num / torch.where(den > 0, den, torch.ones_like(den))
    c = b + wgt * (a - b)
    return torch.where(live, y[n] + q * (s[n] - p * c), torch.zeros_like(c))


def _moments(u):
    """Monomials of degree 0 to 3 of unit vectors, each times the root of its
    multiplicity, so that a degree's moment is a plain sum of squares."""
    x, y, z = u.unbind(1)
    r3, r6, r2 = math.sqrt(3.0), math.sqrt(6.0), math.sqrt(2.0)
    return torch.stack([torch.ones_like(x), x, y, z,
                        x * x, y * y, z * z, r2 * x * y, r2 * x * z, r2 * y * z,
                        x * x * x, y * y * y, z * z * z, r3 * x * x * y, r3 * x * x * z,
                        r3 * x * y * y, r3 * y * y * z, r3 * x * z * z, r3 * y * z * z,
                        r6 * x * y * z], 1)


_DEGREES = [(1, 4), (4, 10), (10, 20)]


def _network(case, w, elem, g):
    act = {"tanh": torch.tanh, "squareplus": lambda v: 0.5 * (v + torch.sqrt(v * v + 4.0))}
    m = MODELS[case["model"]]
    f = act[m["actfn"]]
    e = torch.zeros(g.shape[0], dtype=g.dtype, device=g.device)
    last = len(m["layer_sizes"]) - 1
    for t in range(len(m["symbols"])):
        rows = (elem == t).nonzero()[:, 0]
        h = g[rows]
        for q in range(last + 1):
            z = h @ w["weights_%d_%d" % (t, q)].reshape(h.shape[1], -1) + w["biases_%d_%d" % (t, q)]
            if q == last:
                h = z
            else:
                skip = m.get("use_resnet_dt") and q > 0 and z.shape[1] == h.shape[1]
                h = f(z) + h if skip else f(z)
        e = e.index_put((rows,), h[:, 0])
    return e


def _evaluate(case, w, tab, n, elem, i, j, pos):
    """Energies of atoms 0..n-1 over the pairs (i, j), d = pos[j] - pos[i],
    and per pair the derivative of the energy by d."""
    m = MODELS[case["model"]]
    k, b = m["num_filters"], len(m["symbols"])
    d = pos[j] - pos[i]
    r2 = (d * d).sum(1)
    near = ((r2 < m["rmax"] ** 2) & (r2 > 1e-10)).nonzero()[:, 0]
    i, j, d = i[near], j[near], d[near]
    # the slot of a neighbor: its own element first, then the others in order
    ei, ej = elem[i], elem[j]
    slot = torch.where(ei == ej, torch.zeros_like(ei), torch.where(ej < ei, ej + 1, ej))
    bounds = torch.searchsorted(i, torch.arange(0, n + 4096, 4096, device=i.device))
    energy, grads = [], []
    for q in range(len(bounds) - 1):
        lo = q * 4096
        hi = min(n, lo + 4096)
        if hi <= lo:
            break
        sel = slice(int(bounds[q]), int(bounds[q + 1]))
        dd = d[sel].detach().requires_grad_(True)
        r = dd.norm(dim=1)
        hm = _radial(tab, r)[:, :, None] * _moments(dd / r[:, None])[:, None, :]
        p = torch.zeros((hi - lo) * b, k, 20, dtype=torch.float64, device=i.device)
        p = p.index_add(0, (i[sel] - lo) * b + slot[sel], hm)
        g = torch.stack([p[..., 0]] + [(p[..., u:v] ** 2).sum(-1) for u, v in _DEGREES], -1)
        e = _network(case, w, elem[lo:hi], g.reshape(hi - lo, b * k * 4))
        grads.append(torch.autograd.grad(e.sum(), dd)[0])
        energy.append(e.detach())
    return torch.cat(energy), i, j, d, torch.cat(grads)


def _virial6(d, f):
    """-d (x) F of each pair, xx yy zz xy xz yz."""
    return -torch.stack([d[:, 0] * f[:, 0], d[:, 1] * f[:, 1], d[:, 2] * f[:, 2],
                         d[:, 0] * f[:, 1], d[:, 0] * f[:, 2], d[:, 1] * f[:, 2]], 1)


def _np(**kw):
    return {k: (v.cpu().numpy() if torch.is_tensor(v) else v) for k, v in kw.items()}


def exact(case, seed):
    dev = _device()
    atoms, evals = _atoms(case)
    if atoms * evals > (2000000 if dev.type == "cuda" else 20000):
        return None
    w = _weights(case["model"], dev)
    tab = _table(case["model"], w, dev)
    rc = MODELS[case["model"]]["rmax"]

    def forces(n, elem, i, j, pos, owner):
        e, i, j, d, g = _evaluate(case, w, tab, n, elem[owner], i, j, pos)
        f = torch.zeros(n, 3, dtype=torch.float64, device=dev)
        f = f.index_add(0, i, g).index_add(0, owner[j], -g)
        return e, f, i, _virial6(d, g)

    if case["kind"] == "serve":
        res = []
        for x, types, cell in _requests(case, seed):
            elem = torch.as_tensor(types - 1, device=dev).long()
            e, f, _, v = forces(len(x), elem, *_pairs(x, _box(cell), rc))
            res.append((f, v.sum(0), e.sum()))
        return _np(f=torch.cat([r[0] for r in res]), virial=torch.stack([r[1] for r in res]),
                   energy=torch.stack([r[2] for r in res]))
    x, types, cell, v = _structure(case, seed)
    n = len(x)
    elem = torch.as_tensor(types - 1, device=dev).long()
    if case["kind"] == "list":
        i, j, pos, owner = _pairs(x, _box(cell), rc + SKIN)
        e, i, j, d, g = _evaluate(case, w, tab, n, elem[owner], i, j, pos)
        f = torch.zeros(len(pos), 3, dtype=torch.float64, device=dev)
        f = f.index_add(0, i, g).index_add(0, j, -g)
        vp = _virial6(d, g)
        va = torch.zeros(len(pos), 6, dtype=torch.float64, device=dev)
        va = va.index_add(0, i, 0.5 * vp).index_add(0, j, 0.5 * vp)
        return _np(f=f, eatom=e, vatom=va if case["vatom"] else None, virial=vp.sum(0), energy=e.sum())
    # one pair list with room for the motion of a short segment
    i, j, pos, owner = _pairs(x, _box(cell), rc + 0.8)
    x = torch.as_tensor(x, device=dev)
    shift = pos - x[owner]
    e, f, _, vp = forces(n, elem, i, j, x[owner] + shift, owner)
    if case["kind"] == "static":
        return _np(f=f, eatom=e, virial=vp.sum(0), energy=e.sum())
    mass = torch.as_tensor(np.array(MODELS[case["model"]]["masses"]), device=dev)[elem][:, None]
    mvv2e = 1.0364269e-4
    v = torch.as_tensor(v, device=dev)
    epot, ekin = [], []
    for _ in range(case["steps"]):
        v = v + 0.5 * DT / mvv2e * f / mass
        x = x + DT * v
        e, f, _, vp = forces(n, elem, i, j, x[owner] + shift, owner)
        v = v + 0.5 * DT / mvv2e * f / mass
        epot.append(e.sum())
        ekin.append(0.5 * mvv2e * (mass * v * v).sum())
    return _np(x=x, v=v, f=f, eatom=e, virial=vp.sum(0), epot=torch.stack(epot), ekin=torch.stack(ekin))
