"""Transposed operators on stacked windows: every window gives what it gives
alone, and the cells outside the windows' interiors stay the caller's."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.problems import FAT, random_problem, rel

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-11, "f32": 1e-5}      # twice the parity suite's bars, as for its images and gradients
NZ, NX, NY, NTS, SUB = 27, 31, 79, 4, 4
# first plane, planes and x columns: a gap before, between and behind, one window of the grid's width
WINDOWS = ((1, 25, 26), (29, 21, NX), (51, 23, 22))


def grid(nx, ny):
    return O.Grid(nz=NZ, nx=nx, ny=ny, nts=NTS, sub=SUB, dz=10.0, dx=10.0, dy=10.0, dts=0.002, minPad=4, alphaCos=0.95)


def make_prop(g, precision, graph=False):
    from elasticisolib_3d_amd.propagator import Propagator
    prop = Propagator(g.nz, g.nx, g.ny, g.nts, g.sub, g.dz, g.dx, g.dy, g.dts, g.minPad, g.alphaCos, precision)
    prop.set_gradient_checkpoints(4, 0, "native")
    prop.set_graph(graph)
    return prop


def window_problems(nrec, fluid=()):
    """One problem per window; the upper third of the windows listed in `fluid` has mu = 0."""
    out = []
    for k, (_, ny, nx) in enumerate(WINDOWS):
        g = grid(nx, ny)
        P = random_problem(g, seed=40 + k, nsrc=2, nrec=nrec)
        if k in fluid:
            top = np.zeros(g.shape, bool)
            top[:, :, :NZ // 3] = True
            P["lam"] = np.where(top, P["lam"] + 2 * P["mu"], P["lam"])
            P["mu"] = np.where(top, 0.0, P["mu"])
            P["med"] = O.lib_scale_medium(P["rho"], P["lam"], P["mu"], g.dtw)
        out.append((g, P))
    return out


def box(k):
    y0, ny, nx = WINDOWS[k]
    return np.s_[..., y0:y0 + ny, :nx, :]


def interior():
    m = np.zeros((NY, NX, NZ), bool)
    for y0, ny, nx in WINDOWS:
        m[y0 + FAT:y0 + ny - FAT, FAT:nx - FAT, FAT:NZ - FAT] = True
    return m


def stack(probs, key, fill):
    a = np.full((len(probs[0][1][key]) if key == "med" else 3, NY, NX, NZ), fill)
    for k, (_, P) in enumerate(probs):
        a[box(k)] = P["med"] if key == "med" else np.stack([P["rho"], P["lam"], P["mu"]])
    return a


def stack_points(probs, key):
    out = [[] for _ in range(7)]
    for k, (g, P) in enumerate(probs):
        for j in range(7):
            y, r = np.divmod(P[key][j], g.nx * NZ)
            x, z = np.divmod(r, NZ)
            out[j].append(((y + WINDOWS[k][0]) * NX + x) * NZ + z)
    return [np.concatenate(p) for p in out]


def stack_traces(probs, key):
    return [np.concatenate([P[key][c] for _, P in probs]) for c in range(9)]


def set_windows(prop):
    prop.set_windows(*zip(*WINDOWS))


@pytest.mark.parametrize("device", [False, True])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_born_adjoint_adds_inside_the_windows_only(precision, device):
    """A Born adjoint over the whole grid first (its sums stay in the handle's
    buffer), then with windows onto an image that holds something: each window
    against the oracle and, to the bit, its own propagation; every other cell,
    the windows' own FAT layers included, as the caller left it."""
    import torch
    dt = np.float32 if precision == "f32" else np.float64
    to = (lambda x, t=dt: torch.tensor(np.ascontiguousarray(x, t), device="cuda")) if device else \
        (lambda x, t=dt: np.ascontiguousarray(x, t))
    back = (lambda x: x.cpu().numpy()) if device else (lambda x: x)
    probs = window_problems(nrec=5)
    spos, rpos = stack_points(probs, "spos"), stack_points(probs, "rpos")
    if device:
        spos, rpos = [[torch.tensor(p, device="cuda") for p in q] for q in (spos, rpos)]
    src, rec = [[to(t) for t in stack_traces(probs, k)] for k in ("src", "rec")]
    full = grid(NX, NY)
    prop = make_prop(full, precision)
    prop.set_medium(to(random_problem(full, seed=1)["med"]))
    prop.born_adjoint(spos, src, rec, rpos)
    set_windows(prop)
    prop.set_medium(to(stack(probs, "med", 1.0)))
    # an image of whole numbers times the size of the windows' images, exact in both precisions
    start = np.rint(np.random.default_rng(2).standard_normal((8, NY, NX, NZ)) * 8).astype(dt)
    img = back(prop.born_adjoint(spos, src, rec, rpos, to(start.copy())))
    out = ~interior()
    assert np.array_equal(img[:, out], start[:, out])
    for k, (g, P) in enumerate(probs):
        alone = make_prop(g, precision)
        alone.set_medium(to(P["med"]))
        own = back(alone.born_adjoint(P["spos"], [to(t) for t in P["src"]], [to(t) for t in P["rec"]], P["rpos"],
                                      to(start[box(k)])))
        assert np.array_equal(img[box(k)], own)
        ref = O.lib_born_adjoint(g, P["med"], P["src"], P["spos"], P["rec"], P["rpos"])
        fresh = back(alone.born_adjoint(P["spos"], [to(t) for t in P["src"]], [to(t) for t in P["rec"]], P["rpos"]))
        assert rel(fresh, ref) < TOL[precision]


# receivers per window and list: few (injected in the step's blocks) and many (a launch of their own)
@pytest.mark.parametrize("nrec", [5, 70])
@pytest.mark.parametrize("fluid", [(), (1,), (0, 2), (0, 1, 2)])
@pytest.mark.parametrize("medium,graph", [("scaled", False), ("scaled", True), ("elastic", True)])
def test_transposed_steps_of_a_stack_equal_each_window_alone(medium, graph, fluid, nrec):
    """FP32 gradient, source gradient and Born adjoint of a stack, to the bit
    what each window gives alone: neither the cells outside the windows (zeros
    in a stack of scaled arrays) nor a fluid in another window decides how a
    window's transposed wavefield is held."""
    probs = window_problems(nrec, fluid)
    spos, rpos = stack_points(probs, "spos"), stack_points(probs, "rpos")
    src, rec = stack_traces(probs, "src"), stack_traces(probs, "rec")

    def run(prop, spos, src, rpos, rec):
        data = prop.gradient_forward(spos, src, rpos)
        g8, gs = prop.gradient_backward(spos, src, rpos, rec)
        return data, g8, gs, prop.born_adjoint(spos, src, rec, rpos)

    prop = make_prop(grid(NX, NY), "f32", graph)
    set_windows(prop)
    if medium == "scaled":
        prop.set_medium(stack(probs, "med", 0.0))
    else:
        prop.set_elastic(stack(probs, "elastic", 1.0), probs[0][0].dtw)
    for _ in range(2):   # a repeated call replays the kept graphs
        data, g8, gs, img = run(prop, spos, src, rpos, rec)
        for k, (g, P) in enumerate(probs):
            alone = make_prop(g, "f32", graph)
            if medium == "scaled":
                alone.set_medium(P["med"])
            else:
                alone.set_elastic(np.stack([P["rho"], P["lam"], P["mu"]]), g.dtw)
            d1, g1, s1, i1 = run(alone, P["spos"], P["src"], P["rpos"], P["rec"])
            assert all(np.array_equal(a[nrec * k:nrec * (k + 1)], b) for a, b in zip(data, d1))
            assert all(np.array_equal(a[2 * k:2 * (k + 1)], b) for a, b in zip(gs, s1))
            inner = np.s_[:, FAT:-FAT, FAT:-FAT, FAT:-FAT]
            assert np.array_equal(g8[box(k)][inner], g1[inner])
            assert np.array_equal(img[box(k)][inner], i1[inner])
            ref, sref = O.lib_gradient(g, P["med"], P["src"], P["spos"], P["rec"], P["rpos"])
            assert rel(g1, ref) < TOL["f32"] and rel(s1, sref) < TOL["f32"]
    out = ~interior()
    assert not np.any(g8[:, out]) and not np.any(img[:, out])


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_born_forward_of_a_stack_equals_each_window_alone(precision):
    """Linearised data of a stack, after a call over the whole grid left other
    perturbations in the handle's buffer: each window's own to the bit, and
    the oracle's; perturbations outside the windows are not read."""
    probs = window_problems(5)
    spos, rpos = stack_points(probs, "spos"), stack_points(probs, "rpos")
    src = stack_traces(probs, "src")
    full = grid(NX, NY)
    P = random_problem(full, seed=1)
    prop = make_prop(full, precision)
    prop.set_medium(P["med"])
    prop.born_forward(spos, src, P["dm"], rpos)
    set_windows(prop)
    prop.set_medium(stack(probs, "med", 0.0))
    dm = np.full((8, NY, NX, NZ), np.nan)
    for k, (_, P) in enumerate(probs):
        dm[box(k)] = P["dm"]
    data = prop.born_forward(spos, src, dm, rpos)
    for k, (g, P) in enumerate(probs):
        alone = make_prop(g, precision)
        alone.set_medium(P["med"])
        own = alone.born_forward(P["spos"], P["src"], P["dm"], P["rpos"])
        assert all(np.array_equal(a[5 * k:5 * (k + 1)], b) for a, b in zip(data, own))
        assert rel(own, O.lib_born_forward(g, P["med"], P["src"], P["spos"], P["dm"], P["rpos"])) < TOL[precision]


# z interiors of 32-cell and of 64-cell tiles, both derivative formats, both precisions
@pytest.mark.parametrize("precision,nz,derivatives", [("f64", 27, "native"), ("f32", 27, "s16"), ("f32", 58, "native"),
                                                      ("f32", 58, "s16")])
@pytest.mark.parametrize("medium", ["scaled", "elastic"])
def test_mixed_stack_in_every_kernel(monkeypatch, medium, precision, nz, derivatives):
    """A stack with a fluid in one window, in the kernels the test above does
    not reach and for tile settings of 4, 8 and 16 rows: each window's own
    gradient, source gradient and image to the bit."""
    import sys
    monkeypatch.setattr(sys.modules[__name__], "NZ", nz)
    probs = window_problems(5, (1,))
    spos, rpos = stack_points(probs, "spos"), stack_points(probs, "rpos")
    src, rec = stack_traces(probs, "src"), stack_traces(probs, "rec")

    def run(prop, spos, src, rpos, rec):
        prop.set_gradient_derivatives(derivatives)
        prop.gradient_forward(spos, src, rpos)
        return prop.gradient_backward(spos, src, rpos, rec) + (prop.born_adjoint(spos, src, rec, rpos),)

    own = []
    for g, P in probs:
        alone = make_prop(g, precision)
        alone.set_medium(P["med"]) if medium == "scaled" else \
            alone.set_elastic(np.stack([P["rho"], P["lam"], P["mu"]]), g.dtw)
        own.append(run(alone, P["spos"], P["src"], P["rpos"], P["rec"]))
    prop = make_prop(grid(NX, NY), precision)
    set_windows(prop)
    prop.set_medium(stack(probs, "med", 0.0)) if medium == "scaled" else \
        prop.set_elastic(stack(probs, "elastic", 1.0), probs[0][0].dtw)
    for tile in (None, (4, 3), (8, 5), (16, 8)):
        if tile:
            prop.set_tiling(*tile)
        g8, gs, img = run(prop, spos, src, rpos, rec)
        for k, (g1, s1, i1) in enumerate(own):
            inner = np.s_[:, FAT:-FAT, FAT:-FAT, FAT:-FAT]
            assert all(np.array_equal(a[2 * k:2 * (k + 1)], b) for a, b in zip(gs, s1))
            assert np.array_equal(g8[box(k)][inner], g1[inner]) and np.array_equal(img[box(k)][inner], i1[inner])
