"""Arguments a call must refuse, or take by another route, before any of them
is read."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from tests.problems import random_problem

pytestmark = pytest.mark.gpu

G = O.Grid(nz=20, nx=19, ny=18, nts=4, sub=2, dz=10.0, dx=10.0, dy=10.0, dts=0.001, minPad=3, alphaCos=0.95)


def make_prop(precision="f32"):
    from elasticisolib_3d_amd.propagator import Propagator
    return Propagator(G.nz, G.nx, G.ny, G.nts, G.sub, G.dz, G.dx, G.dy, G.dts, G.minPad, G.alphaCos, precision)


@pytest.mark.parametrize("device", [False, True])
def test_null_trace_arrays_are_refused(device):
    """A component with points but no trace array is an argument error of
    every operator, in host-memory and device-memory calls, and leaves the
    handle usable."""
    import torch
    from elasticisolib_3d_amd import _lib
    P = random_problem(G, seed=3)
    prop = make_prop()
    dev = lambda x, t: torch.tensor(np.asarray(x), dtype=t, device="cuda")  # noqa: E731
    put = (lambda x: dev(x, torch.float32)) if device else (lambda x: np.ascontiguousarray(x, np.float32))
    pos = (lambda x: dev(x, torch.int64)) if device else (lambda x: x)
    spos, rpos = [pos(p) for p in P["spos"]], [pos(p) for p in P["rpos"]]
    src, rec = [put(x) for x in P["src"]], [put(x) for x in P["rec"]]
    prop.set_medium(put(P["med"]))
    want = prop.nl_forward(spos, src, rpos)
    mem = prop._mem_of(*src)
    sp, rp = prop._points(spos, mem), prop._points(rpos, mem)
    field = put(np.zeros((8,) + G.shape))
    g8 = torch.zeros((8,) + G.shape, dtype=torch.float64, device="cuda") if device else np.zeros((8,) + G.shape)
    fp, gp = prop._ptr(field), prop._ptr(g8)
    ref = ctypes.byref
    for comp in (0, 4, 8):
        st, rt = prop._traces(src, prop._counts(spos)), prop._traces(rec, prop._counts(rpos))
        nos, nor = _lib.ElaTraces.from_buffer_copy(st), _lib.ElaTraces.from_buffer_copy(rt)
        nos.tr[comp] = nor.tr[comp] = None
        for s, r in ((nos, rt), (st, nor)):
            prop.gradient_forward(spos, src, rpos)   # the refused gradient_forward below forgets its checkpoints
            a = (ref(sp), ref(s), ref(rp), ref(r), mem)
            b = (ref(sp), ref(s), fp, ref(rp), ref(r), mem)
            g = (ref(sp), ref(s), ref(rp), ref(r), gp, ref(st), mem)
            for name, args in (("nl_forward", a), ("nl_adjoint", a), ("born_forward", b), ("born_adjoint", b),
                               ("gradient_backward", g), ("gradient_forward", a)):
                assert getattr(prop.lib, "ela_" + name)(prop.h, *args) == 1, name   # ELA_ERR_ARG
                assert b"null trace array" in prop.lib.ela_last_error()
        prop.gradient_forward(spos, src, rpos)
        g = (ref(sp), ref(st), ref(rp), ref(rt), gp, ref(nos), mem)
        assert prop.lib.ela_gradient_backward(prop.h, *g) == 1
    again = prop.nl_forward(spos, src, rpos)
    assert all((np.asarray(x.cpu() if device else x) == np.asarray(y.cpu() if device else y)).all()
               for x, y in zip(want, again))


@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_outputs_in_pinned_host_memory(precision):
    """Device-memory calls whose image and gradient lie in pinned host memory,
    which no kernel adds to in place: the same bits as in the GPU's own memory,
    onto what the arrays hold."""
    import torch
    P = random_problem(G, seed=5)
    prop = make_prop(precision)
    prop.set_gradient_checkpoints(2, 0, "native")
    td = torch.float32 if precision == "f32" else torch.float64
    dev = lambda x, t=td: torch.tensor(np.asarray(x), dtype=t, device="cuda")  # noqa: E731
    spos, rpos = [[dev(p, torch.int64) for p in P[k]] for k in ("spos", "rpos")]
    src, rec = [[dev(x) for x in P[k]] for k in ("src", "rec")]
    prop.set_medium(dev(P["med"]))
    prop.gradient_forward(spos, src, rpos)
    mem = prop._mem_of(*src)
    sp, rp = prop._points(spos, mem), prop._points(rpos, mem)
    st, rt = prop._traces(src, prop._counts(spos)), prop._traces(rec, prop._counts(rpos))
    gs = prop._alloc_traces(prop._counts(spos), True)
    gt = prop._traces(gs, prop._counts(spos))
    ref = ctypes.byref
    torch.manual_seed(1)
    held = torch.randn((8,) + G.shape, dtype=td)
    zero = torch.zeros((8,) + G.shape, dtype=torch.float64)   # sums of several segments: equal bits from zero
    out = []
    for pin in (False, True):
        img, g8 = (x.pin_memory() if pin else x.cuda() for x in (held, zero))
        assert prop.lib.ela_born_adjoint(prop.h, ref(sp), ref(st), img.data_ptr(), ref(rp), ref(rt), mem) == 0
        assert prop.lib.ela_gradient_backward(prop.h, ref(sp), ref(st), ref(rp), ref(rt), g8.data_ptr(), ref(gt), mem) == 0
        torch.cuda.synchronize()
        out.append((img.cpu(), g8.cpu()))
    assert all(torch.equal(a, b) for a, b in zip(*out))
    assert float(out[0][1].abs().max()) > 0 and not torch.equal(out[0][0], held)
