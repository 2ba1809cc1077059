"""mdas_run takes its passes through two kernels when nothing wants the phases
apart (no timing, no log, no learned mode) and through one kernel per phase
otherwise.  Both leave the same tree, counters and statistics, also where a
pass is refused for capacity, where the initial grid already meets the
target, and for the single calls that follow a run.  The passes' statistics
come in rows that the kernels write to the host, in turn."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def mdas():
    import pmdas_amd
    from pmdas_amd import kdgrid
    pmdas_amd.load()
    return kdgrid


def _equal(a, b, what):
    for k in a:
        u = a[k].view(np.uint32) if a[k].dtype == np.float32 else a[k]
        v = b[k].view(np.uint32) if b[k].dtype == np.float32 else b[k]
        assert np.array_equal(u, v), (what, k)


# kind, dim, W, H, spp, b, e, alpha, cand, capacity factor, launch shape
# (chunks, error workgroups): one initial leaf, less than a chunk, edges of
# the 64 super groups (64, 65 chunks), several chunks per selection workgroup
CASES = [
    (1, 3, 16, 16, 24, 0, 0, 0.25, 4, 1.6, None),
    (5, 4, 37, 21, 12, 0, 2, 0.5, 1, 1.6, None),
    (3, 5, 64, 48, 8, 1, 2, 0.25, 4, 1.6, None),
    (2, 4, 160, 90, 10, 1, 4, 0.25, 4, 1.6, (64, 64)),
    (3, 5, 160, 90, 10, 1, 4, 0.25, 2, 1.6, (65, 64)),
    (4, 6, 96, 54, 16, 1, 3, 0.125, 8, 1.6, (4096, 1024)),
    (3, 5, 200, 150, 12, 1, 5, 0.25, 4, 1.6, (8192, 8192)),
    (3, 5, 40, 30, 3, 1, 3, 0.25, 4, 4.0, None),    # no pass: the initial grid has 6.8 spp
    (2, 4, 64, 48, 40, 1, 2, 0.0, 4, 1.02, None),   # a pass beyond the capacity
    (3, 5, 64, 48, 20, 1, 2, 0.25, 4, 1.0, None),   # the capacity is the target: the guard ends the run
]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[1]}d-{c[2]}x{c[3]}-{i}" for i, c in enumerate(CASES)])
def test_both_paths_agree(mdas, case):
    import pmdas_amd
    kind, dim, W, H, spp, b, e, alpha, cand, factor, shape = case
    target = spp * W * H
    cap = max(int(target * factor), 4 << (b * dim + 2 * e))
    sc = mdas.Scene(kind, 9, dim, float(W), float(H))
    out = []
    for timed in (False, True):
        _say(f"{case} timed={timed}")
        g = mdas.KDGrid(dim, cap, cand, b, e, alpha, float(W), float(H))
        if shape:
            g.set_launch_shape(*shape)
        g.set_timing(timed)
        rc = 0
        for _ in range(2):  # a second run on the same grid starts over
            try:
                g.Run(sc, target)
            except pmdas_amd.MdasError as err:
                rc = err.code
        st = [g.download_state()]
        info = [rc, g.GetNumberOfSamples(), g.GetNumberOfNodes(), g.GetNewSamples(), g.GetNewNodes(), g.GetMaxError()]
        stats = g.pass_stats()
        # single calls after the run
        try:
            g.AdaptiveSampling()
            g.EvalIntegrand(sc, 0, g.GetNumberOfSamples())
            g.SamplingPass()
        except pmdas_amd.MdasError as err:
            info.append(err.code)
        st.append(g.download_state())
        info += [g.GetNumberOfSamples(), g.GetNumberOfNodes(), g.GetMaxError(), g.Validate()]
        out.append((st, info, stats))
        g.close()
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][2], out[1][2])
    for i, when in enumerate(("run", "after")):
        _equal(out[0][0][i], out[1][0][i], when)


@pytest.mark.parametrize("target", [4, 5, 1000, 4000])
def test_rows_of_runs_batches_and_single_passes(mdas, target):
    """From no pass at all to more passes than there are rows (256), on one
    grid by turns: a batch leaves the rows a run leaves, and single passes and
    another run after either see their own."""
    args = (3, 8000, 4, 0, 0, 1.0, 1.0, 1.0)
    sc = mdas.Scene(1, 3, 3, 1.0, 1.0)
    a, b = mdas.KDGrid(*args), mdas.KDGrid(*args)
    batch = mdas.Batch([b], [sc])
    for turn in range(3):
        passes = a.Run(sc, target)
        batch.run([target])
        rows = a.pass_stats(max_rows=passes + 1)
        assert rows.shape[0] == passes and (passes > 256 or target < 4000)
        assert np.array_equal(rows, b.pass_stats(max_rows=passes + 1))
        assert np.array_equal(rows[1:, 1], rows[:-1, 1] + rows[:-1, 2])
        assert a.GetNumberOfSamples() == (rows[-1, 1] + rows[-1, 2] if passes else 4)
        for _ in range(turn):
            for g in (a, b):
                g.SamplingPass()
                g.EvalNewSamples(sc)
            assert a.GetNewSamples() == b.GetNewSamples() > 0
        _equal(a.download_state(), b.download_state(), (target, turn))
    batch.close()
    for x in (a, b, sc):
        x.close()
