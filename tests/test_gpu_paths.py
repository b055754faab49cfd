"""Paths of the time loop that the structured meshes do not take (needs an
MI355X), against the oracle bit for bit: points with more than four element
copies, solid points coupled to several fluid points, other numbers of linear
solids than five, several source elements, sources in the fluid, fields in
several pieces.  The meshes are those of test_gpu_synthetic, changed.
"""
import numpy as np
import pytest
import torch

import fluid_source
import perf.cases as C
import test_gpu_synthetic as T

pytestmark = pytest.mark.gpu

TINY = dict(nth=21, nm=7, nf=3, ni=2, rec=15)


def _changed(monkeypatch, mesh=None, state=None):
    """The meshes and states of perf.cases passed through mesh, state."""
    if mesh:
        def build(case):
            M = C._build_mesh(*(case[k] for k in ("nth", "nm", "nf", "ni", "colat", "scheme",
                                                  "anel", "aniso")))
            mesh(M)
            return M
        monkeypatch.setattr(C, "_mesh", build)
    if state:
        plain = C._state
        monkeypatch.setattr(C, "_state", lambda *a: state(plain(*a)))


# ---------------------------------------------------------------------------
# points that the structured grid does not have
# ---------------------------------------------------------------------------
def _join(M, dom, pairs):
    """Points b become points a of region dom (pairs of a, b)."""
    g = M[dom]
    gid = g["gid"].clone()
    for a, b in pairs:
        gid[gid == b] = a
    keep, inv = torch.unique(gid, return_inverse=True)
    g["gid"], g["n"] = inv.reshape(gid.shape), len(keep)
    g["xy"] = [v[keep] for v in g["xy"]]
    g["axpt"] = g["axpt"][keep]
    if "gamma" in g:
        g["gamma"] = g["gamma"][keep]
    rho = g["rho"] if dom == "s" else 1 / (g["rho"] * g["vp"] ** 2)
    g["mass"] = C._assemble(g["gid"], g["n"], g["W"] * rho)


def _points(M, dom, copies, elements):
    """Points off the axis and off the solid-fluid boundary with so many
    copies, in the elements."""
    g = M[dom]
    n = torch.bincount(g["gid"].reshape(-1), minlength=g["n"])
    ok = (n == copies) & ~g["axpt"]
    e, j = (M["bse"], M["bjs"]) if dom == "s" else (M["bfe"], M["bjf"])
    ok[g["gid"][e, j].reshape(-1)] = False
    ids = torch.unique(g["gid"][elements])
    return ids[ok[ids]].tolist()


def _boundary(M, dom, a, b):
    """Vertices (two copies, off the axis) of boundary entries a .. b - 1."""
    g = M[dom]
    e, j = (M["bse"], M["bjs"]) if dom == "s" else (M["bfe"], M["bjf"])
    n = torch.bincount(g["gid"].reshape(-1), minlength=g["n"])
    ids = torch.unique(g["gid"][e[a:b], j[a:b]])
    return ids[(n[ids] == 2) & ~g["axpt"][ids]].tolist()


def _outer(M):
    return slice(0, 3 * M["nth"])                 # solid elements numbered first


def _inner(M):
    return slice(7 * M["nth"], None)              # and last


def _eight(M):
    v = _points(M, "s", 4, _outer(M))
    _join(M, "s", [(v[3], v[-4])])


def _five(M):
    _join(M, "s", [(_points(M, "s", 4, _outer(M))[5], _points(M, "s", 1, _inner(M))[2])])


def _coupled_first(M):
    _join(M, "s", [(_boundary(M, "s", 2, 9)[1], _points(M, "s", 4, _inner(M))[3])])


def _coupled_last(M):
    _join(M, "s", [(_points(M, "s", 4, _outer(M))[3], _boundary(M, "s", 2, 9)[1])])


def _fluid_eight(M):
    v = _points(M, "f", 4, slice(None))
    _join(M, "f", [(v[1], v[-2])])


def _fluid_coupled(M):
    _join(M, "f", [(_boundary(M, "f", 2, 9)[1], _points(M, "f", 4, slice(None))[-2])])


def _two_fluid_points(M):
    v = _boundary(M, "s", 2, 9)
    _join(M, "s", [(v[0], v[2])])


def _all(M):
    for change in (_eight, _fluid_eight, _coupled_first, _two_fluid_points):
        change(M)


# where the fluid is assembled by a launch of its own before the solid
SPLIT = {_coupled_last, _fluid_coupled, _two_fluid_points, _all}


@pytest.mark.parametrize("change", [_eight, _five, _coupled_first, _coupled_last, _fluid_eight,
                                    _fluid_coupled, _two_fluid_points, _all],
                         ids=lambda f: f.__name__[1:])
def test_points_of_many_copies(change, tmp_path, monkeypatch):
    print("mesh:", change.__name__, flush=True)
    _changed(monkeypatch, mesh=change)
    for src, o in (("0", {}), ("1", dict(scheme=1, anel=1)), ("2", dict(anel=2)),
                   ("111", dict(scheme=1)), ("00", dict(anel=1))):
        T._check(tmp_path, src, (3, 4), graph=2, **o)
    T._check(tmp_path, "1", (3, 4), colat=60, **dict(scheme=1))
    case = dict(C._BASE, **TINY)
    s, _, _ = T._member(case, C._mesh(case), C, 0, 1, str(tmp_path / "p.bin"))
    s.set_profiling(True)
    s.run(2)
    assert s.kernel_stats()["fluid_assemble_update"][1] == (2 if change in SPLIT else 0)
    s.close()


# ---------------------------------------------------------------------------
# linear solids, sources
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("ns", [1, 4, 6, 8])
def test_numbers_of_linear_solids(ns, tmp_path, monkeypatch):
    def solids(M):
        om = 2 * np.pi / (M["dt"] * np.geomspace(40.0, 10000.0, ns))
        E = np.exp(-om * M["dt"])
        q = (1 - E) / (om * M["dt"])
        aj = M["aj"][:, :1] * torch.linspace(1, 0.3, ns, dtype=C.F8, device=C.DEV)
        M.update(ns=ns, expw=E, tst=1 - q, tstm1=q - E, aj=aj.contiguous())

    _changed(monkeypatch, mesh=solids)
    for anel in (1, 2):
        for scheme in (0, 1):
            for src in ("0", "1", "2", "11", "2222"):
                T._check(tmp_path, src, (3, 3), scheme=scheme, anel=anel)


@pytest.mark.parametrize("scheme", [0, 1])
def test_several_source_elements(scheme, tmp_path, monkeypatch):
    """Eight elements, two by four, with terms at the points they share."""
    seed = iter(range(100))

    def sources(st):
        gid = st["igloc_solid"].reshape(-1, 25)
        els = np.array([layer * TINY["nth"] + col for layer in range(1, 5) for col in (3, 4)])
        n, own = np.bincount(gid.ravel()), np.bincount(gid[els].ravel(), minlength=gid.max() + 1)
        rng = np.random.default_rng(next(seed))
        val = rng.standard_normal((3, gid.max() + 1)) * np.abs(st["source_term"]).max()
        val *= (n == own) & (n > 0)              # all of the point's copies are in the block
        if st.dims["src_type"] == 0:
            val[1] = 0
        assert np.count_nonzero(val[0]) == 7 * 15
        t = val[:, gid[els]].astype(np.float32).ravel()
        st.arrays["source_term"] = (t, (t.size,))
        st.arrays["ielsrc"] = ((els + 1).astype(np.int32), (8,))
        st.dims["nelsrc"] = 8
        return st

    _changed(monkeypatch, state=sources)
    for src in ("0", "1", "2", "00", "111", "2222"):
        T._check(tmp_path, src, (3, 4), scheme=scheme, anel=1)


def test_sources_in_the_fluid(tmp_path, monkeypatch):
    _changed(monkeypatch, state=lambda st: fluid_source.fluid_source_state(
        st, fluid_source.pick_fluid_elements(st)))
    for src, o in (("0", {}), ("1", dict(anel=1)), ("2", dict(anel=2)), ("00", {}), ("111", {}),
                   ("0012", {}), ("0", dict(colat=60))):
        T._check(tmp_path, src, (3, 4), graph=2, **o)


# ---------------------------------------------------------------------------
# fields and snapshots in pieces
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("nth,nm,pieces", [(21, 7, 1), (64, 24, 2), (100, 36, 3)])
def test_downloaded_fields_in_pieces(nth, nm, pieces, tmp_path):
    """Expanded by the GPU into 2**18 floats at a time, of a wavefield alone
    and of a member of a group, against the fields uploaded and the oracle."""
    case = dict(C._BASE, nth=nth, nm=nm, nf=4, ni=3, rec=5)
    mesh = C._mesh(case)
    members = [T._member(case, mesh, C, 1, q, str(tmp_path / ("s%d.bin" % q))) for q in (1, 2)]
    total = 25 * (6 * nth * (nm + 3) + 3 * nth * 4)
    assert -(-total // (1 << 18)) == pieces
    for s, o, d in members:
        before = s.fields()                      # not yet run: copied and expanded on the host
        s.run(0)
        for a, b, c in zip(before, s.fields(), o.fields()):
            T._bits(a, b)
            T._bits(a, c)
        s.run(2)
        o.run(1, 2, 5, d["seis_it"])
        for a, b in zip(s.fields(), o.fields()):
            T._bits(a, b)
        # some of the fields only
        f = [np.zeros_like(a) for a in before]
        s._ok(s._L.axh_download_fields(s._h, None, _ptr(f[1]), None, None, _ptr(f[4])))
        T._bits(f[1], o.fields()[1])
        T._bits(f[4], o.fields()[4])
    with T.Batch([m[0] for m in members]) as b:
        b.run(1)
        for s, o, d in members:
            o.run(3, 3, 5, d["seis_it"])
            for a, c in zip(s.fields(), o.fields()):
                T._bits(a, c)
    for s, _, _ in members:
        s.close()


def _ptr(a):
    return a.ctypes.data


@pytest.mark.parametrize("ring", [0, 2, 3])
@pytest.mark.parametrize("scheme,graph", [(0, 0), (0, 8), (1, 2)])
def test_snapshot_rings(scheme, graph, ring, tmp_path):
    """A snapshot every other step, the ring shorter than the run; a ring too
    short for the snapshots of a graph launches directly."""
    case = dict(C._BASE, **TINY, src="1", scheme=scheme, strain_it=2)
    s, o, d = T._member(case, C._mesh(case), C, 1, 100, str(tmp_path / "s.bin"))
    s.set_kwf(strain_it=2, ring_snapshots=ring)
    s.set_graph_steps(graph)
    got = [s.run_kwf(n) for n in (19, 4, 17)]
    want, snaps = T._oracle_run(o, d, 40, 2)
    T._bits(np.concatenate([g[0] for g in got]), want)
    T._bits(np.concatenate([g[1] for g in got]), snaps)
    s.close()
