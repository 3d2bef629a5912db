"""Fields to the host in one piece, in several with a ragged last one, and
without a pinned buffer: the same bytes, and no device memory for it.  A
request's reservation covers its model."""
import ctypes as C

import numpy as np
import pytest

from test_adv2d_resident_gpu import _model as adv2d_model
from test_hpe_gpu import _pair as hpe_pair
from test_sw2d_resident_gpu import _model as sw2d_model

pytestmark = pytest.mark.gpu


def _sw2d():
    m = sw2d_model(N=5, nX=9, nY=7, precision="fp64")
    m.ForwardStepRK3(0.0, 1)
    return m


def _adv2d():
    return adv2d_model(N=4, nX=9, nY=7, nq=3)


def _hpe():
    m = hpe_pair(dict(N=3, n=(3, 2, 5), periodic=(False, True), warp=0.02, dp=True), dt=2e-3)[1]
    m.ForwardStepRK3(1)
    return m


@pytest.mark.parametrize("make", [_sw2d, _adv2d, _hpe])
def test_every_way_gives_the_same_bytes(gpu_lib, make, monkeypatch):
    m = make()
    monkeypatch.setenv("SELF_AMD_STAGE_DOUBLES", "0")
    want = m.GetSolution()
    assert np.isfinite(want).all() and want.any()
    for most in ("1", "700", "1000000"):  # an element a piece, a few, all
        monkeypatch.setenv("SELF_AMD_STAGE_DOUBLES", most)
        assert np.array_equal(m.GetSolution(), want), most
    monkeypatch.delenv("SELF_AMD_STAGE_DOUBLES")
    assert np.array_equal(m.GetSolution(), want)


@pytest.mark.parametrize("N,nX,nY", [(2, 70, 70), (6, 30, 30), (7, 34, 21)])
def test_large_arrays_at_every_alignment(gpu_lib, N, nX, nY):
    """From 1 MB on an array is written past the caches, in 16-byte stores with
    8-byte ones at a row's ends: rows of odd and even lengths, the caller's
    array on and off 16 bytes and off 8, nothing beside it touched."""
    L = gpu_lib
    m = sw2d_model(N=N, nX=nX, nY=nY, precision="fp64")
    m.ForwardStepRK3(0.0, 1)
    want = np.ascontiguousarray(m.GetSolution()).ravel()
    assert want.nbytes >= 1 << 20 and np.isfinite(want).all()
    buf = np.empty(want.nbytes + 64, np.uint8)
    first = -buf.ctypes.data % 16 + 16
    for off in (first, first + 8, first + 4):
        buf[:] = 0xa5
        L.check(L.lib().self_sw2d_get_field(m._h, 0, C.cast(buf.ctypes.data + off, L.dp)))
        got = buf[off:off + want.nbytes]
        assert np.array_equal(got, want.view(np.uint8))
        assert (buf[:off] == 0xa5).all() and (buf[off + want.nbytes:] == 0xa5).all()
    m.Trash()


def test_reading_a_field_takes_no_device_memory(gpu_lib):
    m = _sw2d()
    before = m.DeviceBytes()
    m.GetSolution()
    assert m.DeviceBytes() == before


def test_an_array_of_nodes_goes_there_and_back(gpu_lib, monkeypatch):
    from test_cgsem_resident_gpu import _model as cgsem_model
    m = cgsem_model(5, 9, 7, boundary=True)
    rng = np.random.default_rng(3)
    for most in (None, "0", "1", "700"):
        if most is not None:
            monkeypatch.setenv("SELF_AMD_STAGE_DOUBLES", most)
        u = rng.standard_normal(m.mesh.x.shape)
        m.SetSolution(u)
        got = m.GetSolution()
        monkeypatch.setenv("SELF_AMD_STAGE_DOUBLES", "0")
        assert np.array_equal(m.GetSolution(), got)
        monkeypatch.delenv("SELF_AMD_STAGE_DOUBLES")
        inner = u[:, 1:-1, 1:-1]  # nodes of one element each
        assert np.array_equal(got[:, 1:-1, 1:-1], inner)
        m.SetSolution(got)  # copies of a shared node agree now, so this changes nothing
        assert np.array_equal(m.GetSolution(), got)
    m.Trash()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("nX,N", [(32, 7), (64, 3)])
def test_a_request_reserves_what_its_model_holds(gpu_lib, precision, nX, N):
    """The server's models launch their stages from the host: they allocate no
    buffers of the resident form.  Built here with the server's calls."""
    from self_amd import _lib as L
    from self_amd import serving as S
    lib, check = L.lib(), L.check
    srv = S.Server(workers=1)
    spec = S.make_inputs(S.Spec(S.REQ_SW2D, nX, N, 7, precision, 2))
    res, out = srv.wait(srv.submit(spec))
    srv.close()
    assert res.status == 0 and np.isfinite(out).all()
    m = sw2d_model(N=N, nX=nX, nY=nX, precision=precision)
    h, held = C.c_void_p(), C.c_size_t()
    d = L.SWDesc(N, m.nElems, m.mesh.nEdges, {"fp64": L.FP64, "mixed": L.MIXED}[precision], L.FUSED, 1.0, 1e-4, 0.0)
    check(lib.self_sw2d_create(C.byref(d), C.byref(h)))
    check(lib.self_sw2d_set_graph(h, 0))
    g, ns = m.mesh, m.dgStorage
    check(lib.self_sw2d_set_nodal(h, L.ptr(ns.flat("dMatS")), L.ptr(ns.flat("dMatP")), L.ptr(ns.qWeight),
                                  L.ptr(ns.qWeight), L.ptr(ns.lagWest), L.ptr(ns.lagEast), L.ptr(ns.lagSouth),
                                  L.ptr(ns.lagNorth)))
    check(lib.self_sw2d_set_geometry(h, L.ptr(g.edges, L.ip), L.ptr(g.dxds), L.ptr(g.dxdp), L.ptr(g.dyds),
                                     L.ptr(g.dydp), L.ptr(g.J), L.ptr(g.nHat), L.ptr(g.nLen)))
    sol = np.ascontiguousarray(m.GetSolution())
    check(lib.self_sw2d_set_field(h, 0, L.ptr(sol)))
    check(lib.self_sw2d_forward_step_rk3(h, 0.0, 4))
    check(lib.self_sw2d_get_field(h, 0, L.ptr(sol)))
    check(lib.self_sw2d_device_bytes(h, C.byref(held)))
    check(lib.self_sw2d_destroy(h))
    nodes = g.nElems * (N + 1) ** 2
    resident = 3 * 8 * nodes + 2 * 16 * g.nElems * 8 * (N + 1) + 4  # second state, messages, status
    m.GetSolution()
    assert m.DeviceBytes() == held.value + resident
    assert held.value <= res.bytes
    m.Trash()
