"""Injection inside a step's own blocks and recording by the step after
(few points) against the separate injection launch (many points) and the FP64
oracle, at tile edges and the smallest records."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.problems import random_problem, rel

pytestmark = pytest.mark.gpu

TOL = {"f64": 1e-11, "f32": 5e-6}      # the parity suite's bars
# interior 70 x 9 x 11: two z tiles (64 + 6 cells), three x tiles of 4 rows, several y chunks
NZ, NX, NY = 78, 17, 19


def grid(nts, sub):
    return O.Grid(nz=NZ, nx=NX, ny=NY, nts=nts, sub=sub, dz=10.0, dx=10.0, dy=10.0, dts=0.0005 * sub, minPad=3,
                  alphaCos=0.95)


def edge_points():
    """Both sides of every tile edge and the interior's corners."""
    zs, xs, ys = (4, 67, 68, NZ - 5), (4, 7, 8, NX - 5), (4, 5, 6, 11, 12, NY - 5)
    return np.array([(y * NX + x) * NZ + z for y in ys for x in xs for z in zs], np.int64)


def make_prop(g, precision):
    from elasticisolib_3d_amd.propagator import Propagator
    return Propagator(g.nz, g.nx, g.ny, g.nts, g.sub, g.dz, g.dx, g.dy, g.dts, g.minPad, g.alphaCos, precision)


# points per list: 9 (few, one box), 56 (504 over the 9 components: still in the blocks), 57 (513: separate launch)
@pytest.mark.parametrize("n", [9, 56, 57])
@pytest.mark.parametrize("precision,nts,sub,graph", [("f64", 2, 1, False), ("f64", 3, 3, False), ("f64", 4, 2, True),
                                                     ("f64", 3, 6, False), ("f64", 3, 7, False),
                                                     ("f32", 3, 4, True), ("f32", 3, 2, False)])
def test_points_in_the_steps_blocks(n, precision, nts, sub, graph):
    g = grid(nts, sub)
    P = random_problem(g, seed=5 + n)
    pts = edge_points()
    P["spos"] = [np.roll(pts, 7 * k)[:n] for k in range(7)]
    P["rpos"] = [np.roll(pts, 11 * k + 3)[:n] for k in range(7)]
    rng = np.random.default_rng(n)
    P["src"] = [rng.standard_normal((n, nts)) * 1e3 for _ in range(9)]
    P["rec"] = [rng.standard_normal((n, nts)) for _ in range(9)]
    prop = make_prop(g, precision)
    prop.set_graph(graph)
    prop.set_elastic(np.stack([P["rho"], P["lam"], P["mu"]]), g.dtw)
    med = P["med"]
    fwd, adj = (O.lib_nl_forward(g, med, P["src"], P["spos"], P["rpos"]),
                O.lib_nl_adjoint(g, med, P["rec"], P["spos"], P["rpos"]))
    for _ in range(2):   # a repeated call replays the kept graph
        assert rel(prop.nl_forward(P["spos"], P["src"], P["rpos"]), fwd) < TOL[precision]
        assert rel(prop.nl_adjoint(P["spos"], P["rec"], P["rpos"]), adj) < TOL[precision]
    prop.set_gradient_checkpoints(2, 0, "native")
    g8_ref, gs_ref = O.lib_gradient(g, med, P["src"], P["spos"], P["rec"], P["rpos"])
    rec = prop.gradient_forward(P["spos"], P["src"], P["rpos"])
    assert rel(rec, fwd) < TOL[precision]
    g8, gs = prop.gradient_backward(P["spos"], P["src"], P["rpos"], P["rec"])
    assert rel(g8, g8_ref) < 2 * TOL[precision] and rel(gs, gs_ref) < 2 * TOL[precision]
    if nts >= 3:
        born = O.lib_born_forward(g, med, P["src"], P["spos"], P["dm"], P["rpos"])
        assert rel(prop.born_forward(P["spos"], P["src"], P["dm"], P["rpos"]), born) < TOL[precision]
        img = O.lib_born_adjoint(g, med, P["src"], P["spos"], P["rec"], P["rpos"])
        assert rel(prop.born_adjoint(P["spos"], P["src"], P["rec"], P["rpos"]), img) < TOL[precision]


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_fused_and_separate_injection_give_the_same_bits(precision):
    """The tile shape decides whether a list's box is small enough for the
    blocks (8 rows and 24 planes: at most 1024 tiles meet it; 4 rows and
    single planes: more do), and the results do not depend on it."""
    nz, nx, ny, nts, sub = 140, 90, 60, 3, 2
    g = O.Grid(nz=nz, nx=nx, ny=ny, nts=nts, sub=sub, dz=10.0, dx=10.0, dy=10.0, dts=0.001, minPad=4, alphaCos=0.95)
    P = random_problem(g, seed=3)
    corner = np.array([(y * nx + x) * nz + z for y in (4, ny - 5) for x in (4, nx - 5) for z in (4, nz - 5)], np.int64)
    pos = [corner] * 7
    src = [np.random.default_rng(1).standard_normal((8, nts)) * 1e3 for _ in range(9)]
    prop = make_prop(g, precision)
    prop.set_elastic(np.stack([P["rho"], P["lam"], P["mu"]]), g.dtw)
    out = []
    for tx, yc in ((8, 24), (4, 1)):
        prop.set_tiling(tx, yc)
        out.append(prop.nl_forward(pos, src, pos) + [prop.born_adjoint(pos, src, src, pos)])
    assert all(np.array_equal(a, b) for a, b in zip(*out))


# z interiors of one 32-cell tile, one cell more, a ragged last tile, and one
# where FP32 keeps the 64-cell tiles; x interiors below, at and past 8 rows
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("iz,ix", [(32, 8), (33, 9), (90, 7), (64, 17), (1, 1)])
def test_narrow_tiles(precision, iz, ix):
    """32 x 8 tiles (4 rows set) against 64 x 8 tiles bit for bit, and the
    oracle, for the forward, the gradient (derivative store and paired
    imaging) and the Born pair."""
    g = O.Grid(nz=iz + 8, nx=ix + 8, ny=17, nts=3, sub=4, dz=10.0, dx=10.0, dy=10.0, dts=0.002, minPad=2, alphaCos=0.95)
    P = random_problem(g, seed=iz, nsrc=1, nrec=1)
    prop = make_prop(g, precision)
    prop.set_elastic(np.stack([P["rho"], P["lam"], P["mu"]]), g.dtw)
    prop.set_gradient_checkpoints(4, 0, "native")
    out = []
    for tx, yc in ((4, 3), (8, 4)):
        prop.set_tiling(tx, yc)
        rec = prop.gradient_forward(P["spos"], P["src"], P["rpos"])
        g8, gs = prop.gradient_backward(P["spos"], P["src"], P["rpos"], P["rec"])
        out.append([*rec, g8, *gs, *prop.nl_adjoint(P["spos"], P["rec"], P["rpos"]),
                    *prop.born_forward(P["spos"], P["src"], P["dm"], P["rpos"]),
                    prop.born_adjoint(P["spos"], P["src"], P["rec"], P["rpos"])])
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    fwd = O.lib_nl_forward(g, P["med"], P["src"], P["spos"], P["rpos"])
    g8_ref, gs_ref = O.lib_gradient(g, P["med"], P["src"], P["spos"], P["rec"], P["rpos"])
    assert rel(rec, fwd) < TOL[precision]
    assert rel(g8, g8_ref) < 2 * TOL[precision] and rel(gs, gs_ref) < 2 * TOL[precision]


# 16 points x 300 samples: packed (173 kB of receiver traces); x 1000: past the packed size, copied array by array
@pytest.mark.parametrize("nts", [300, 1000])
def test_host_traces_packed_and_direct(nts):
    """Host-memory calls against the same call on device tensors, bit for
    bit, for trace blocks that travel in one pinned copy and larger ones."""
    import torch
    g = O.Grid(nz=20, nx=19, ny=18, nts=nts, sub=1, dz=10.0, dx=10.0, dy=10.0, dts=0.0005, minPad=3, alphaCos=0.95)
    P = random_problem(g, seed=9, nsrc=2, nrec=16)
    prop = make_prop(g, "f32")
    prop.set_elastic(np.stack([P["rho"], P["lam"], P["mu"]]), g.dtw)
    dev = lambda xs, dt: [torch.tensor(np.asarray(x), dtype=dt, device="cuda") for x in xs]  # noqa: E731
    sp, rp = dev(P["spos"], torch.int64), dev(P["rpos"], torch.int64)
    src, rec = dev(P["src"], torch.float32), dev(P["rec"], torch.float32)
    for _ in range(2):
        pairs = [(prop.nl_forward(P["spos"], P["src"], P["rpos"]), prop.nl_forward(sp, src, rp)),
                 (prop.nl_adjoint(P["spos"], P["rec"], P["rpos"]), prop.nl_adjoint(sp, rec, rp))]
        for host, device in pairs:
            assert all(np.array_equal(a, b.cpu().numpy()) for a, b in zip(host, device))


# mu / (lambda + 2 mu) of the upper half: as drawn, a fluid, a soft solid, and on both sides of the rule's 2^-20
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("ratio", [None, 0.0, 0.01, 0.9e-6, 3e-6])
def test_transposed_wavefield_kinds(precision, ratio):
    """The transposed steps hold M n alone for the velocities and shear stresses
    of a solid medium and n beside it otherwise: Born adjoint, gradient and
    source gradient against the oracle on both sides of the rule, both medium
    kinds, after a switch of the medium on one handle."""
    g = grid(4, 4)
    P = random_problem(g, seed=21, nsrc=2, nrec=9)
    lam, mu = P["lam"].copy(), P["mu"].copy()
    if ratio is not None:
        top = np.zeros(g.shape, bool)
        top[:, :, :NZ // 2] = True
        p = lam + 2 * mu
        mu = np.where(top, ratio * p, mu)
        lam = p - 2 * mu
    med = O.lib_scale_medium(P["rho"], lam, mu, g.dtw)
    img = O.lib_born_adjoint(g, med, P["src"], P["spos"], P["rec"], P["rpos"])
    g8_ref, gs_ref = O.lib_gradient(g, med, P["src"], P["spos"], P["rec"], P["rpos"])
    prop = make_prop(g, precision)
    prop.set_gradient_checkpoints(4, 0, "native")
    prop.set_medium(P["med"])
    prop.born_adjoint(P["spos"], P["src"], P["rec"], P["rpos"])
    for kind in ("scaled", "elastic"):
        if kind == "scaled":
            prop.set_medium(med)
        else:
            prop.set_elastic(np.stack([P["rho"], lam, mu]), g.dtw)
        out = prop.born_adjoint(P["spos"], P["src"], P["rec"], P["rpos"])
        prop.gradient_forward(P["spos"], P["src"], P["rpos"])
        g8, gs = prop.gradient_backward(P["spos"], P["src"], P["rpos"], P["rec"])
        e = rel(out, img), rel(g8, g8_ref), rel(gs, gs_ref)
        print(f"{precision} ratio {ratio} {kind}: image {e[0]:.2e} gradient {e[1]:.2e} source gradient {e[2]:.2e}", flush=True)
        assert e[0] < 2 * TOL[precision] and e[1] < 2 * TOL[precision] and e[2] < 2 * TOL[precision]


# densities of a rigid body: 1 / M overflows in FP32, M n underflows, and both still fit
@pytest.mark.parametrize("precision", ["f64", "f32"])
@pytest.mark.parametrize("rho", [1e36, 1e32, 1e12])
def test_transposed_steps_in_a_rigid_body(precision, rho):
    """A block whose buoyancies are next to nothing: n is not recovered from
    M n there. Born adjoint and gradient against the oracle, every array by
    itself (the buoyancies' hold the block's cells)."""
    g = grid(4, 4)
    P = random_problem(g, seed=27, nsrc=2, nrec=9)
    r = P["rho"].copy()
    r[6:12, 6:11, 30:50] = rho
    med = O.lib_scale_medium(r, P["lam"], P["mu"], g.dtw)
    img = O.lib_born_adjoint(g, med, P["src"], P["spos"], P["rec"], P["rpos"])
    g8_ref, gs_ref = O.lib_gradient(g, med, P["src"], P["spos"], P["rec"], P["rpos"])
    prop = make_prop(g, precision)
    prop.set_gradient_checkpoints(4, 0, "native")
    prop.set_elastic(np.stack([r, P["lam"], P["mu"]]), g.dtw)
    out = prop.born_adjoint(P["spos"], P["src"], P["rec"], P["rpos"])
    prop.gradient_forward(P["spos"], P["src"], P["rpos"])
    g8, gs = prop.gradient_backward(P["spos"], P["src"], P["rpos"], P["rec"])
    e = [rel(a, b) for a, b in zip([*out, *g8], [*img, *g8_ref])] + [rel(gs, gs_ref)]
    print(f"{precision} rho {rho:g}: worst array {max(e):.2e}", flush=True)
    assert np.all(np.isfinite(out)) and np.all(np.isfinite(g8)) and max(e) < 2 * TOL[precision]


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_velocity_tile_direction(precision):
    """Velocity tiles run backwards where the layers of y chunks are small
    and forwards where they are not (600-plane chunks): the same bits, and the
    oracle's data, with sources in the step's blocks."""
    g = grid(3, 4)
    P = random_problem(g, seed=33, nsrc=5, nrec=9)
    out = []
    for planes in (4, 600):
        prop = make_prop(g, precision)
        prop.set_tiling(4, planes)
        prop.set_elastic(np.stack([P["rho"], P["lam"], P["mu"]]), g.dtw)
        out.append(prop.nl_forward(P["spos"], P["src"], P["rpos"]))
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    assert rel(out[0], O.lib_nl_forward(g, P["med"], P["src"], P["spos"], P["rpos"])) < TOL[precision]
