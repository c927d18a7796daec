"""The work a user of the engine has it do, as cases that can be timed and compared.

A program holds closed curves on the host (arrays, or a BCC file), and wants
their certificate: the curves go to the GPU (`set_curves_packed` or
`load_bcc`), spline curves become polylines (`discretize_current`), the pairs
that could be linked are found (`potential_links`) and their linking numbers
computed (`linking_numbers`), by the direct sum or by Barnes-Hut with the beta
or the learned criterion.  A simulation repeats all of it with new positions
every step (upload = True); a program that keeps its curves on the GPU and asks
again, with another method or for a check, repeats the last two calls
(upload = False).  Besides that a user trains the learned criterion.

The models are those of the repository's benchmark (fastlinkingnumbers_amd/
workloads.py, the same geometry, drawn here on the GPU because that is quicker):
ten loops with a Hopf and a torus link, sheets of chain mail, rings on a helical
lattice, and pairs of interlinked random walks, from a few hundred vertices to
sixteen million.
"""
import math
import os
import struct
import tempfile

import numpy as np
import torch

import fastlinkingnumbers_amd as flk
from fastlinkingnumbers_amd import criterion, workloads

TAU = 2 * math.pi
# Pairs of a hybrid certificate below this many segment pairs are summed
# directly, as in the benchmark's lattice workload.
HYBRID = 4096 * 4096
# Results are kept in arrays of one size whatever the number of candidate
# pairs, which differs from one set of positions to the next: this many rows
# for each curve (a ring of a lattice touches about seven others' boxes, half
# of them counted with it), and no fewer than MIN_ROWS.
ROWS_PER_CURVE = 8
MIN_ROWS = 64
# exact() sums at most this many segment pairs (about 10 s).
EXACT_MOST = 1.2e10


def listed():
    """Smallest to largest, each path and type that a program uses."""
    return [
        # ten short loops, direct sum: the smallest certificate, all latency
        dict(name="ten loops direct 200", kind="certificate", model="ten", n=200, dtype="float64",
             method="directsum", criterion="beta", fp64=0, threshold=0, upload=True),
        # ten loops of the benchmark's size and the default method
        dict(name="ten loops barneshut 2000", kind="certificate", model="ten", n=2000, dtype="float64",
             method="barneshut", criterion="beta", fp64=0, threshold=0, upload=True),
        # a knit-sized sheet, every step new positions, direct sum
        dict(name="chainmail direct 12x12", kind="certificate", model="chainmail", grid=12, nmin=64, nmax=2048,
             dtype="float32", method="directsum", criterion="beta", fp64=0, threshold=0, upload=True),
        # a sheet with FP64 coordinates summed in FP64, the check of a result
        dict(name="chainmail fp64 16x16", kind="certificate", model="chainmail", grid=16, nmin=64, nmax=16384,
             dtype="float64", method="directsum", criterion="beta", fp64=1, threshold=0, upload=False),
        # the benchmark's headline sheet: curves resident, candidate pairs and direct sum
        dict(name="chainmail direct 40x40", kind="certificate", model="chainmail", grid=40, nmin=256, nmax=65536,
             dtype="float32", method="directsum", criterion="beta", fp64=0, threshold=0, upload=False),
        # many small trees, the default method
        dict(name="lattice barneshut 400", kind="certificate", model="lattice", loops=400, nmin=64, nmax=4096,
             dtype="float32", method="barneshut", criterion="beta", fp64=0, threshold=0, upload=True),
        # short and long loops together: direct sums beside Barnes-Hut
        dict(name="lattice hybrid 1000", kind="certificate", model="lattice", loops=1000, nmin=64, nmax=262144,
             dtype="float32", method="barneshut", criterion="beta", fp64=0, threshold=HYBRID, upload=True),
        # one pair of long tangled curves, three sizes, both criteria
        dict(name="walks beta 30k", kind="certificate", model="walks", n=30011, dtype="float32",
             method="barneshut", criterion="beta", fp64=0, threshold=0, upload=True),
        dict(name="walks beta 2M", kind="certificate", model="walks", n=2000000, dtype="float32",
             method="barneshut", criterion="beta", fp64=0, threshold=0, upload=True),
        dict(name="walks learned 8M", kind="certificate", model="walks", n=8000000, dtype="float32",
             method="barneshut", criterion="mlp", fp64=0, threshold=0, upload=True),
        # a BCC file of splines: read, discretize, certificate
        dict(name="splines 24x24", kind="splines", grid=24, nmin=64, nmax=8192, method="barneshut"),
        # training of the learned criterion, forward and backward
        dict(name="train 65k", kind="train", n=65536, batch=8192, epochs=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges; sizes log-uniform, so odd ones mostly."""
    what = rng.choice(["ten", "chainmail", "chainmail fp64", "lattice", "lattice hybrid", "walks", "walks learned",
                       "splines", "train"])
    upload = rng.random() < 0.7
    cert = dict(kind="certificate", dtype=rng.choice(["float32", "float64"]), method="barneshut", criterion="beta",
                fp64=0, threshold=0, upload=upload)
    if what == "ten":
        return dict(cert, model="ten", n=_log_int(rng, 100, 4000), method=rng.choice(["directsum", "barneshut"]))
    if what == "chainmail":
        return dict(cert, model="chainmail", grid=rng.randint(3, 30), nmin=rng.randint(16, 256),
                    nmax=_log_int(rng, 512, 30000), method="directsum")
    if what == "chainmail fp64":
        return dict(cert, model="chainmail", grid=rng.randint(3, 18), nmin=rng.randint(16, 256),
                    nmax=_log_int(rng, 512, 16384), method="directsum", fp64=1)
    if what == "lattice":
        return dict(cert, model="lattice", loops=_log_int(rng, 20, 2000), nmin=rng.randint(16, 256),
                    nmax=_log_int(rng, 512, 16384))
    if what == "lattice hybrid":
        return dict(cert, model="lattice", loops=_log_int(rng, 50, 900), nmin=rng.randint(16, 256),
                    nmax=_log_int(rng, 8192, 262144), threshold=HYBRID)
    if what == "walks":
        return dict(cert, model="walks", n=_log_int(rng, 1000, 4000000))
    if what == "walks learned":
        return dict(cert, model="walks", n=_log_int(rng, 10000, 7000000), criterion="mlp", dtype="float32")
    if what == "splines":
        return dict(kind="splines", grid=rng.randint(3, 24), nmin=rng.randint(16, 128), nmax=_log_int(rng, 256, 8192),
                    method=rng.choice(["directsum", "barneshut"]))
    return dict(kind="train", n=_log_int(rng, 5000, 100000), batch=rng.choice([1024, 4096, 8192]), epochs=1)


# ---------------------------------------------------------------- models
def _sizes(g, count, nmin, nmax):
    return np.rint(np.exp(g.uniform(np.log(nmin), np.log(nmax), size=count))).astype(np.int64)


def _rot45(sign):
    a = np.array([1.0, 1.0, 0.0]) / np.sqrt(2.0)
    k = np.array([[0, -a[2], a[1]], [a[2], 0, -a[0]], [-a[1], a[0], 0]])
    s = sign * np.pi / 4
    return np.eye(3) + np.sin(s) * k + (1 - np.cos(s)) * (k @ k)


def _rings(n, frame, centre, radial, axial):
    """Rings of n[c] vertices: (r cos t, r sin t, w) in frame[c] (its columns
    the images of the axes) about centre[c], with r = 1 + sum a cos(f t + p)
    over the modes in radial (arrays a, f, p of shape (modes, rings)) and
    w = sum a sin(f t + p) over those in axial.  A (total, 3) FP64 GPU tensor."""
    up = lambda a: torch.as_tensor(np.asarray(a, dtype=np.float64), device="cuda")  # noqa: E731
    sizes = torch.as_tensor(n, device="cuda")
    c = torch.repeat_interleave(torch.arange(len(n), device="cuda"), sizes)
    first = torch.cumsum(sizes, 0) - sizes
    t = (torch.arange(len(c), device="cuda") - first[c]).double() * TAU / sizes[c]
    r, w = torch.ones_like(t), torch.zeros_like(t)
    for a, f, p in zip(*map(up, radial)):
        r += a[c] * torch.cos(f[c] * t + p[c])
    for a, f, p in zip(*map(up, axial)):
        w += a[c] * torch.sin(f[c] * t + p[c])
    x, y = r * torch.cos(t), r * torch.sin(t)
    f, o = up(frame), up(centre)
    return torch.stack([o[c, d] + f[c, d, 0] * x + f[c, d, 1] * y + f[c, d, 2] * w for d in range(3)], 1)


def _chainmail(seed, grid, nmin, nmax):
    """A sheet of rings tilted +-45 degrees, each linked with its neighbours."""
    g = np.random.default_rng([2, seed])
    m = grid * grid
    n = _sizes(g, m, nmin, nmax)
    i, j = np.divmod(np.arange(m), grid)
    frame = np.where(((i + j) % 2 == 0)[:, None, None], _rot45(1), _rot45(-1))
    centre = np.stack([1.5 * i, 1.5 * j, np.zeros(m)], 1)
    none = (np.zeros((0, m)),) * 3
    wave = (np.full((1, m), 0.05), g.integers(3, 8, size=(1, m)), g.uniform(0, TAU, size=(1, m)))
    return _rings(n, frame, centre, none, wave), n


def _lattice(seed, loops, nmin, nmax, per_turn=101, pitch=1.6, amp=0.1):
    """The sheet wrapped into a tube, three random modes on each ring."""
    g = np.random.default_rng([4, seed])
    n = _sizes(g, loops, nmin, nmax)
    k = np.arange(loops)
    th, z = TAU * k / per_turn, pitch * k / per_turn
    e_t = np.stack([-np.sin(th), np.cos(th), 0 * th], 1)
    e_r = np.stack([np.cos(th), np.sin(th), 0 * th], 1)
    e_z = np.stack([0 * th, 0 * th, 1 + 0 * th], 1)
    sheet = np.where((k % 2 == 0)[:, None, None], _rot45(1), _rot45(-1))
    frame = np.stack([e_t, e_z, e_r], 2) @ sheet
    centre = per_turn * pitch / TAU * e_r + z[:, None] * e_z
    modes = lambda: (g.uniform(0, amp / 3, size=(3, loops)), g.integers(2, 7, size=(3, loops)),  # noqa: E731
                     g.uniform(0, TAU, size=(3, loops)))
    return _rings(n, frame, centre, modes(), modes()), n


def _walks(seed, n):
    """Two closed Gaussian random walks about nearly the same centre.  The
    steps are summed as whole numbers, so the same seed gives the same bits."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rg = 100.0 * math.sqrt(n / 2e6)  # the benchmark's density at any length
    out = []
    for k in range(2):
        s = (torch.randn(3, n, device="cuda", generator=gen) * 2.0 ** 20).round().to(torch.int64)
        x = torch.cumsum(s, 1)
        end, mean = x[:, -1:].double(), x.sum(1, keepdim=True).double() / n
        i = torch.arange(n, device="cuda", dtype=torch.float64) / n
        x = (x.double() - i * end - (mean - end * ((n - 1) / (2 * n)))).T
        x *= rg / (2.0 ** 20 * math.sqrt(n / 4.0))
        if k:
            d = np.random.default_rng([5, seed]).normal(size=3)
            x += torch.as_tensor(0.25 * rg * d / np.linalg.norm(d), device="cuda")
        out.append(x)
    return torch.cat(out), np.array([n, n], dtype=np.int64)


def _curves(case, seed):
    """Packed vertices on the host (FP32 values, or FP64 ones that FP32 cannot
    hold) and the offsets."""
    if case["model"] == "ten":
        cs = workloads.hopf_torus_circles(seed, n_circle=case["n"], n_torus=2 * case["n"])
        n = np.array([len(c) for c in cs], dtype=np.int64)
        x = torch.as_tensor(np.concatenate(cs))
    elif case["model"] == "chainmail":
        x, n = _chainmail(seed, case["grid"], case["nmin"], case["nmax"])
    elif case["model"] == "lattice":
        x, n = _lattice(seed, case["loops"], case["nmin"], case["nmax"])
    else:
        x, n = _walks(seed, case["n"])
    dtype = torch.float32 if case["dtype"] == "float32" else torch.float64
    return x.to(dtype).contiguous().cpu().numpy(), np.concatenate([[0], np.cumsum(n)])


# ---------------------------------------------------------------- the three programs
class _State:
    pass


def prepare(case, seed):
    st = _State()
    st.kind = case["kind"]
    st.engine = flk.Engine(0)
    if st.kind == "train":
        g = np.random.default_rng([6, seed])
        st.params, st.norm = criterion.load_weights()
        mean, std = st.norm[:flk.MLP_NFEAT], st.norm[flk.MLP_NFEAT:]
        z = g.standard_normal((case["n"], flk.MLP_NFEAT), dtype=np.float32)
        st.x = (mean + std * z).astype(np.float32)
        st.y = (_network(st.params, z) + 0.5 * g.standard_normal(case["n"], dtype=np.float32)).astype(np.float32)
        st.params = criterion.init_params(seed)
        st.batch, st.epochs, st.seed = case["batch"], case["epochs"], seed % 1000
        return st
    if st.kind == "splines":
        # control polygons of cubic B-splines in a BCC file, as a knit model comes
        x, n = _chainmail(seed, case["grid"], case["nmin"], case["nmax"])
        st.folder = tempfile.TemporaryDirectory()
        st.path = os.path.join(st.folder.name, "model.bcc")
        _write_bcc(st.path, x.float().cpu().numpy(), n)
        st.params = flk.default_params(method=case["method"])
    else:
        st.xyz, st.offsets = _curves(case, seed)
        st.upload = case["upload"]
        st.params = flk.default_params(method=case["method"], criterion=case["criterion"], fp64=case["fp64"],
                                       bh_direct_threshold=case["threshold"])
        if case["criterion"] == "mlp":
            st.engine.mlp_set_weights(*criterion.load_weights())
        if not st.upload:
            st.engine.set_curves_packed(st.xyz, st.offsets)
    torch.cuda.empty_cache()
    return st


def run(st):
    eng = st.engine
    if st.kind == "train":
        eng.mlp_set_weights(st.params, st.norm)
        loss = eng.mlp_train(st.x, st.y, epochs=st.epochs, batch=st.batch, lr=2e-3, seed=st.seed)
        return {"weights": eng.mlp_get_weights()[0], "loss": np.float32(loss)}
    out = {}
    if st.kind == "splines":
        info = eng.load_bcc(st.path)
        links = eng.potential_links()  # boxes of the control polygons hold the splines
        d = eng.discretize_current(info["segment_type"], info["looped"], links)
        out["discretized"] = np.array([d["rounds"], d["segments"], d["pieces"], d["vertices"], *d["overlaps"]])
        out["boxes"] = eng.curve_boxes()
    elif st.upload:
        eng.set_curves_packed(st.xyz, st.offsets)
    pairs = eng.potential_links()
    res = eng.linking_numbers(pairs, st.params)
    cert = np.array(flk.certificate_from_lk(pairs, res.lk), dtype=np.int64).reshape(-1, 3)
    rows = max(MIN_ROWS, ROWS_PER_CURVE * eng.ncurves)
    out["count"] = np.array([len(pairs), len(cert)])
    out["pairs"], out["certificate"] = _kept(pairs, rows), _kept(cert, rows)
    out["lk"], out["err"], out["flags"] = _kept(res.lk, rows), _kept(res.err, rows), _kept(res.flags, rows, np.int64)
    return out


def _kept(a, rows, dtype=None):
    out = np.zeros((rows,) + a.shape[1:], dtype=dtype or a.dtype)
    out[:len(a)] = a
    return out


def _write_bcc(path, xyz, n):
    head = struct.pack("<3sB2sBBQQ40s", b"BCC", 0x44, b"BS", 3, 2, len(n), int(n.sum()), b"")
    with open(path, "wb") as f:
        f.write(head)
        at = 0
        for k in n:
            f.write(struct.pack("<i", -int(k)))
            f.write(xyz[at:at + k].tobytes())
            at += k


def _network(p, z):
    """The 12-64-64-1 hard-swish network on normalised features, FP32 host."""
    h = lambda v: v * np.clip(v / 6 + 0.5, 0, 1)  # noqa: E731
    a = h(z @ p[:768].reshape(64, 12).T + p[768:832])
    a = h(a @ p[832:4928].reshape(64, 64).T + p[4928:4992])
    return a @ p[4992:5056] + p[5056]


# ---------------------------------------------------------------- what a pass cannot do without
def _mean_size(nmin, nmax):
    return (nmax - nmin) / math.log(nmax / nmin) if nmax > nmin else float(nmin)


def work(case):
    if case["kind"] == "train":
        # 12-64-64-1 forward, and twice that backward
        flops = 3 * 2 * (12 * 64 + 64 * 64 + 64) * case["n"] * case["epochs"]
        return {"bytes": 4 * (flk.MLP_NFEAT + 1) * case["n"] + 8 * flk.MLP_NPARAM, "flops": flops}
    if case["kind"] == "splines":
        verts = case["grid"] ** 2 * _mean_size(case["nmin"], case["nmax"])
        # a cubic's exact box and point per segment, then the polyline's tree
        return {"bytes": 2 * 12 * verts, "flops": 1000 * verts}
    if case["model"] == "ten":
        verts, seg_pairs = 12 * case["n"], 5 * case["n"] ** 2
    elif case["model"] == "walks":
        verts, seg_pairs = 2 * case["n"], case["n"] ** 2
    else:
        loops = case["grid"] ** 2 if case["model"] == "chainmail" else case["loops"]
        mean = _mean_size(case["nmin"], case["nmax"])
        verts, seg_pairs = loops * mean, 3.8 * loops * mean ** 2
    size = 4 if case["dtype"] == "float32" else 8
    if case["method"] == "directsum":
        flops = 58 * seg_pairs
    elif case["threshold"]:
        flops = 1000 * verts + 0.1 * 58 * seg_pairs * min(1.0, case["threshold"] / _mean_size(case["nmin"], case["nmax"]) ** 2)
    else:
        # about 470 operations for each visited pair of nodes
        visits = (40 if case["criterion"] == "beta" else 10) if case["model"] == "walks" else 2
        flops = 470 * visits * verts
    return {"bytes": 3 * size * verts, "flops": flops}


# ---------------------------------------------------------------- the same in 64 bits
def _gauss_sum(p, q):
    """Linking integral of two closed polylines ((n, 3), (m, 3) FP64 GPU
    tensors): the solid angles of both triangles of each segment pair's
    quadrilateral (Van Oosterom and Strackee 1983), over 4 pi."""
    if len(p) < len(q):
        p, q = q, p
    p, q = torch.cat([p, p[:1]]), torch.cat([q, q[:1]])
    rows = max(1, 2_000_000 // len(q))
    dot = lambda u, v: (u[0] * v[0] + u[1] * v[1]) + u[2] * v[2]  # noqa: E731
    total = 0.0
    for r in range(0, len(p) - 1, rows):
        s = p[r:r + rows + 1]
        g = [q[None, :, d] - s[:, None, d] for d in range(3)]
        l = torch.sqrt(dot(g, g))
        cut = lambda i, j: ([v[i:i + len(s) - 1, j:j + len(q) - 1] for v in g],  # noqa: E731
                            l[i:i + len(s) - 1, j:j + len(q) - 1])
        (a, la), (b, lb), (c, lc), (d, ld) = cut(0, 0), cut(1, 0), cut(1, 1), cut(0, 1)
        ac = dot(a, c)
        x = [a[1] * c[2] - a[2] * c[1], a[2] * c[0] - a[0] * c[2], a[0] * c[1] - a[1] * c[0]]
        # the triangles (a, b, c) and (a, c, d), counter-clockwise alike
        w1 = torch.atan2(-dot(b, x), la * lb * lc + dot(a, b) * lc + ac * lb + dot(b, c) * la)
        w2 = torch.atan2(dot(d, x), la * lc * ld + ac * ld + dot(a, d) * lc + dot(c, d) * la)
        total += float((w1 + w2).sum())
    return total / TAU


def exact(case, seed):
    """The linking integrals of the candidate pairs in 64 bits, where that is
    quick; the estimate, the flags and a training's weights have no such value."""
    if case["kind"] != "certificate":
        return None
    xyz, off = _curves(case, seed)
    n = np.diff(off)
    x = torch.as_tensor(xyz, device="cuda").double()
    lo = np.array([x[a:b].amin(0).cpu().numpy() for a, b in zip(off[:-1], off[1:])])
    hi = np.array([x[a:b].amax(0).cpu().numpy() for a, b in zip(off[:-1], off[1:])])
    i, j = np.triu_indices(len(n), 1)
    near = np.all((lo[i] <= hi[j]) & (lo[j] <= hi[i]), axis=1)
    i, j = i[near], j[near]
    if float(np.sum(n[i] * n[j])) > EXACT_MOST:
        return None
    lk = [_gauss_sum(x[off[a]:off[a + 1]], x[off[b]:off[b + 1]]) for a, b in zip(i, j)]
    out = dict.fromkeys(["count", "pairs", "certificate", "err", "flags"])
    out["lk"] = _kept(np.array(lk), max(MIN_ROWS, ROWS_PER_CURVE * len(n)))
    return out
