"""Which runs replay graphs of steps (needs an MI355X): by the number of
launches that a graph holds, the mesh and the caller; the results are the
oracle's bit for bit either way (the synthetic meshes of test_gpu_synthetic).
"""
import numpy as np
import pytest

import test_gpu_synthetic as T
from axisem_amd import solver as S
from axisem_amd import tune

pytestmark = pytest.mark.gpu


def _replays(monkeypatch, tmp_path, src, chunks, graph, **options):
    """The replays of each chunk, run and compared by test_gpu_synthetic."""
    seen = []

    def counted(cls, *names):
        def method(name):
            def call(self, *a):
                r = getattr(cls, name)(self, *a)
                seen.append(self.last_run_replays())
                return r
            return call
        return type(cls.__name__, (cls,), {n: method(n) for n in names})

    monkeypatch.setattr(T, "Solver", counted(S.Solver, "run", "run_kwf"))
    monkeypatch.setattr(T, "Batch", counted(S.Batch, "run", "step_kwf"))
    T._check(tmp_path, src, chunks, graph=graph, **options)
    return seen


NEWMARK, SYMPLEC4 = dict(scheme=0), dict(scheme=1)


@pytest.mark.parametrize("src,graph,replayed,options", [
    # newmark2: 2 launches a step, 3 with memory variables at all points or
    # with absorbing boundaries
    ("0", 8, True, NEWMARK), ("0", 9, True, NEWMARK), ("1", 7, False, NEWMARK),
    ("2", 8, True, dict(anel=1)), ("2", 7, False, dict(anel=1)),
    ("1", 6, True, dict(anel=2)), ("2", 7, True, dict(anel=2)), ("0", 5, False, dict(anel=2)),
    ("1", 6, True, dict(colat=60)), ("1", 5, False, dict(colat=60)),
    # symplec4: 8, with the receivers or the memory variables 9; absorbing 13
    ("0", 2, True, SYMPLEC4), ("1", 1, False, SYMPLEC4),
    ("1", 3, True, dict(scheme=1, anel=1)), ("2", 2, True, dict(scheme=1, anel=2)),
    ("0", 3, True, dict(scheme=1, anel=2)), ("2", 2, True, dict(scheme=1, colat=60)),
    # kernel wavefields: in the assembly (newmark2) or a launch of their own
    ("1", 8, True, dict(strain_it=3)), ("1", 9, True, dict(strain_it=2, anel=1)),
    ("0", 2, True, dict(scheme=1, strain_it=3)),
    ("2", 2, True, dict(scheme=1, anel=1, strain_it=2)),
    # one group of wavefields; groups side by side
    ("00", 8, True, NEWMARK), ("111", 7, False, NEWMARK), ("2222", 2, True, SYMPLEC4),
    ("1111", 2, True, dict(scheme=1, anel=2)), ("0012", 1, True, NEWMARK),
])
def test_replayed_or_direct(src, graph, replayed, options, tmp_path, monkeypatch):
    print("graphs of %d steps:" % graph, src, options, flush=True)
    chunks = (2 * graph + 1, graph, max(graph - 1, 1))
    got = _replays(monkeypatch, tmp_path, src, chunks, graph, **options)
    assert got == [n // graph if replayed else 0 for n in chunks]


def test_large_meshes_replay_from_40_launches(tmp_path):
    """8 100 elements: graphs of 19 newmark2 steps are launched directly, of
    20 replayed."""
    import perf.cases as C

    case = dict(C._BASE, nth=100, nm=70, nf=8, ni=3, rec=15, src="0")
    mesh = C._mesh(case)
    runs = []
    for graph in (0, 19, 20):
        s, _, _ = T._member(case, mesh, C, 0, 7, str(tmp_path / "s.bin"))
        s.set_graph_steps(graph)
        runs.append((s.run(41), s.last_run_replays(), s.fields()))
        s.close()
    assert [r[1] for r in runs] == [0, 0, 2]
    for r in runs[1:]:
        T._bits(r[0], runs[0][0])
        for a, b in zip(r[2], runs[0][2]):
            T._bits(a, b)


def _one(tmp_path, **options):
    import perf.cases as C

    case = dict(C._BASE, nth=21, nm=7, nf=3, ni=2, rec=15, src="1", **options)
    return T._member(case, C._mesh(case), C, 1, 100, str(tmp_path / "s.bin"))


def test_queued_runs_replay(tmp_path):
    """axh_run_begin and axh_run_kwf_begin replay graphs of any length."""
    s, o, d = _one(tmp_path, strain_it=3)
    s.set_graph_steps(2)
    seis = [s.run_begin(5)]
    s.run_end()
    assert s.last_run_replays() == 2
    more, kwf = s.run_kwf_begin(6)
    s.run_end()
    assert s.last_run_replays() == 3
    seis += [more, s.run(3)]
    assert s.last_run_replays() == 0
    want, snaps = T._oracle_run(o, d, 14, 3)
    T._bits(np.concatenate(seis), want)
    T._bits(kwf, snaps[2:4])     # of steps 6 and 9
    for a, b in zip(s.fields(), o.fields()):
        T._bits(a, b)
    s.close()


@pytest.mark.parametrize("graph,replays", [(7, 0), (8, 3)])
def test_no_alloc_runs_replay(graph, replays, tmp_path):
    s, o, d = _one(tmp_path)
    s.set_graph_steps(graph)
    got = [s.run(3)]
    out = np.zeros((25, d["num_rec"], 3), np.float32)
    n = S.library().axh_seis_samples(s._h, 4, 28)
    S._check(S.library().axh_run_noalloc(s._h, 4, 28, S._p(out)))
    s.iter = 28
    assert s.last_run_replays() == replays
    T._bits(np.concatenate(got + [out[:n]]), o.run(1, 28, d["num_rec"], d["seis_it"]))
    s.close()


def test_tuner_times_each_schedule_once(tmp_path):
    """Candidates that the library launches directly are the direct schedule."""
    s, _, _ = _one(tmp_path)
    s.close()
    t = tune.tune_solo(str(tmp_path / "s.bin"), steps=16)
    assert set(t["ms_per_step"]) == {0, 8, 16, 32} and t["graph_steps"] in t["ms_per_step"]
    t = tune.tune_solo(str(tmp_path / "s.bin"), steps=16, candidates=(2, 4))
    assert set(t["ms_per_step"]) == {0} and t["graph_steps"] == 0
    t = tune.tune_batch([str(tmp_path / "s.bin")] * 2, steps=16, widths=(2,))
    assert set(t["ms_per_step"]) == {"2/0", "2/8", "2/16", "2/32"}
