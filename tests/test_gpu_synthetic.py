"""GPU time loop against the oracle on the synthetic meshes of perf/cases.py
(needs an MI355X; no recorded state and no host program): every launch form of
a step, from fields in which every point moves, bit for bit.

21 x 12 elements: ragged tiles, axial elements, both solid-fluid boundaries,
and with colat 60 the absorbing boundaries (fluid and solid assembled by two
launches).
"""
import numpy as np
import pytest

from axisem_amd.solver import Batch, BlowUp, Solver
from axisem_amd.state import write_state
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def _member(case, mesh, C, src, seed, path):
    w = C._wave(case, mesh, src, seed)
    w["stf"] = w["stf"][:4000]
    st = C._state(case, mesh, src, w)
    st.dims.update(niter=900, seis_it=1 + seed % 2)
    write_state(st, path)
    so, fl = mesh["s"], mesh["f"]
    el = lambda v, g: v[..., g["gid"]].cpu().numpy().reshape(-1)  # noqa: E731
    fields = [el(w[k], so) for k in ("disp", "velo")] + \
             [el(w[k], fl) for k in ("chi", "dchi", "ddchi")]
    s, o = Solver.from_state_file(path), Oracle(path)
    if case["strain_it"]:
        s.kwf_grid(1, 3, 1, 3)
        s.set_kwf(strain_it=case["strain_it"])
    s.set_fields(*fields)
    o.set_fields(*fields)
    return s, o, st.dims


def _oracle_run(o, d, n, strain_it):
    if not strain_it:
        return o.run(1, n, d["num_rec"], d["seis_it"]), None
    grid = o.kwf_grid(1, 3, 1, 3)
    kwf, seis = [o.kwf_sample(grid, True)], []
    for it in range(1, n + 1):
        seis.append(o.run(it, it, d["num_rec"], d["seis_it"]))
        if it % strain_it == 0:
            kwf.append(o.kwf_sample(grid, True))
    return np.concatenate(seis), np.stack(kwf)


def _bits(a, b):
    np.testing.assert_array_equal(np.asarray(a).view(np.int32), np.asarray(b).view(np.int32))


def _check(tmp_path, srcs, chunks, graph=0, width=4, **options):
    import perf.cases as C

    case = dict(C._BASE, nth=21, nm=7, nf=3, ni=2, rec=15, src=srcs, **options)
    mesh = C._mesh(case)
    members = [_member(case, mesh, C, int(c), 100 + b, str(tmp_path / ("s%d.bin" % b)))
               for b, c in enumerate(srcs)]
    solvers = [m[0] for m in members]
    run = Batch(solvers, group_width=width, graph_steps=graph) if len(srcs) > 1 else solvers[0]
    if len(srcs) == 1:
        run.set_graph_steps(graph)
    seis, kwf = [[] for _ in srcs], [[] for _ in srcs]
    for n in chunks:
        if case["strain_it"]:
            a, k = run.step_kwf(n) if len(srcs) > 1 else run.run_kwf(n)
            for q, x in enumerate(k if len(srcs) > 1 else [k]):
                kwf[q].append(x)
        else:
            a = run.run(n)
        for q, x in enumerate(a if len(srcs) > 1 else [a]):
            seis[q].append(x)
    for q, (s, o, d) in enumerate(members):
        want, snaps = _oracle_run(o, d, sum(chunks), case["strain_it"])
        _bits(np.concatenate(seis[q]), want)
        if snaps is not None:
            _bits(np.concatenate(kwf[q]), snaps)
        for a, b in zip(s.fields(), o.fields()):
            _bits(a, b)
    if len(srcs) > 1:
        run.close()
    for s in solvers:
        s.close()


@pytest.mark.parametrize("anel", [0, 1, 2])
@pytest.mark.parametrize("scheme", [0, 1])
@pytest.mark.parametrize("src", "012")
def test_one_wavefield(src, scheme, anel, tmp_path):
    """Direct launches and replayed graphs of an even and an odd number of
    steps, in chunks with steps left over; closed and absorbing boundaries."""
    o = dict(scheme=scheme, anel=anel)
    _check(tmp_path, src, (3, 1, 4), **o)
    _check(tmp_path, src, (9, 1, 5), graph=3 if anel else 4, **o)
    _check(tmp_path, src, (3, 2), colat=60, aniso=True, **o)


@pytest.mark.parametrize("anel", [0, 1, 2])
@pytest.mark.parametrize("scheme", [0, 1])
def test_batches(scheme, anel, tmp_path):
    """Groups of every width, mixed source types, kernel wavefields."""
    o = dict(scheme=scheme, anel=anel)
    _check(tmp_path, "0012", (5, 4), graph=2, **o)
    _check(tmp_path, "11111", (5, 2), **o)
    _check(tmp_path, "000", (5, 5), graph=4, width=3, **o)
    _check(tmp_path, "222", (5, 5), graph=3, width=2, colat=60, **o)
    _check(tmp_path, "1", (7, 6), graph=2, strain_it=3, **o)
    _check(tmp_path, "00", (4, 5), width=2, strain_it=2, **o)


@pytest.mark.parametrize("anel", [0, 1])
@pytest.mark.parametrize("scheme,steps", [(0, 20), (0, 21), (1, 5), (1, 6)])
def test_replays_of_one_wavefield(scheme, steps, anel, tmp_path):
    """Graphs of just enough launches to be replayed, and one step fewer."""
    o = dict(scheme=scheme, anel=anel)
    _check(tmp_path, "1", (2 * steps + 1, 2, steps), graph=steps, **o)
    _check(tmp_path, "0", (2 * steps,), graph=steps - 1, **o)


def test_more_samples_than_a_run_stages(tmp_path):
    """1100 receivers, 80 and 20 steps: above and below the staged samples."""
    import perf.cases as C

    case = dict(C._BASE, nth=21, nm=7, nf=3, ni=2, rec=1100, src="0", steps=1)
    s, o, d = _member(case, C._mesh(case), C, 0, 100, str(tmp_path / "s.bin"))
    got = np.concatenate([s.run(80), s.run(20)])
    _bits(got, o.run(1, 100, d["num_rec"], d["seis_it"]))
    s.close()


def test_blow_up_is_of_its_own_run(tmp_path):
    """A run that blows up names its step; the next run starts without it."""
    import perf.cases as C

    case = dict(C._BASE, nth=21, nm=7, nf=3, ni=2, rec=15, src="0")
    s, o, d = _member(case, C._mesh(case), C, 0, 100, str(tmp_path / "s.bin"))
    quiet = [np.zeros_like(f) for f in s.fields()]
    loud = [q.copy() for q in quiet]
    loud[0][2 * loud[0].size // 3:] = 1e22
    for _ in range(2):
        at = s.iter + 1
        s.set_fields(*loud)
        with pytest.raises(BlowUp, match="time step %d$" % at):
            s.run(3)
        s.set_fields(*quiet)
        s.run(4)
        assert 0 < s.last_run_ms() < 1000
    s.close()


@pytest.mark.parametrize("graph", [0, 20])
def test_no_alloc_runs(graph, tmp_path):
    """axh_run_noalloc, whose step base, flag and ring are shared and not
    cleared by the last run, between runs of the context's own."""
    import perf.cases as C
    from axisem_amd import solver as S

    case = dict(C._BASE, nth=21, nm=7, nf=3, ni=2, rec=15, src="0")
    s, o, d = _member(case, C._mesh(case), C, 0, 100, str(tmp_path / "s.bin"))
    s.set_graph_steps(graph)
    got = [s.run(3)]
    for n in (21, 2, 22):
        out = np.zeros((n, d["num_rec"], 3), np.float32)
        S._check(S.library().axh_run_noalloc(s._h, s.iter + 1, s.iter + n, S._p(out)))
        s.iter += n
        got += [out, s.run(1)]
        assert 0 < s.last_run_ms() < 1000
    _bits(np.concatenate(got), o.run(1, s.iter, d["num_rec"], d["seis_it"]))
    s.close()
