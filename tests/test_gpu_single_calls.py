"""The single calls (ComputeErrors, AdaptiveSampling, SamplingPass) on trees
that the host did not see grow: uploaded states, down to none, against the
oracle."""
import numpy as np
import pytest

from oracle import pyoracle

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


@pytest.fixture(scope="module")
def mdas():
    import pmdas_amd
    from pmdas_amd import kdgrid
    pmdas_amd.load()
    return kdgrid


@pytest.mark.parametrize("dim", [3, 5])
@pytest.mark.parametrize("samples", [0, 7])
def test_passes_over_no_leaf(mdas, dim, samples):
    """An uploaded state may have no leaf: a pass then adds nothing."""
    _say(f"no leaf dim={dim} samples={samples}")
    g = mdas.KDGrid(dim, 4096, 4, 0, 1, 0.25, 8.0, 8.0)
    sc = mdas.Scene(0, 1, dim, 8.0, 8.0)
    for turn in range(2):
        g.upload_state(np.zeros((samples, dim)), np.zeros((samples, 3)), np.zeros((0, 4)), np.zeros((0, 2 * dim)),
                       np.zeros(0), np.zeros(0))
        for call in (g.SamplingPass, g.ComputeErrors, g.AdaptiveSampling, g.SamplingPass):
            call()
            assert (g.GetNumberOfSamples(), g.GetNumberOfNodes()) == (samples, 0)
            assert (g.GetNewSamples(), g.GetNewNodes(), g.GetMaxError()) == (0, 0, 0.0)
        # the grid is as good as new
        g.InitialSampling()
        g.EvalNewSamples(sc)
        g.SamplingPass()
        assert g.GetNewSamples() > 0
    g.close()
    sc.close()


@pytest.mark.parametrize("dim,kind", [(3, 1), (5, 3)])
@pytest.mark.parametrize("g_error", [np.nan, -np.nan, -1.0, -0.0, 0.0, 1e-45, 1e-3, np.inf])
def test_selection_against_an_uploaded_g_error(mdas, dim, kind, g_error):
    """AdaptiveSampling takes g_error as uploaded, whatever it is: against a
    NaN or a negative one no leaf is selected, against 0 every leaf."""
    _say(f"g_error {g_error} dim={dim}")
    args = (dim, 20000, 4, 0, 2, 0.25, 48.0, 32.0)
    o = pyoracle.OracleGrid(*args)
    o.run(pyoracle.make_scene(kind, 5, dim, 48.0, 32.0), 3000)
    o.compute_errors()
    st = o.state()
    o.set_state(st, g_error)
    o.adaptive_sampling()
    g = mdas.KDGrid(*args)
    g.upload_state(*[st[k] for k in ("coords", "values", "idx", "box", "err", "seed")], g_error)
    assert np.float32(g.GetMaxError()).tobytes() == np.float32(g_error).tobytes()
    g.AdaptiveSampling()
    added = o.n_samples - len(st["coords"])
    assert added == {"nan": 0, "-1.0": 0, "-0.0": 0, "0.0": len(st["idx"]), "inf": added}.get(str(g_error), added)
    assert (g.GetNumberOfSamples(), g.GetNumberOfNodes()) == (o.n_samples, o.n_leaves)
    a, b = g.download_state(), o.state()
    for k in b:
        n = len(st["values"]) if k == "values" else None  # the new ones are not evaluated
        assert np.array_equal(a[k][:n].view(np.uint32), b[k][:n].view(np.uint32)), k
    g.close()
    o.close()


def _check(g, o, what):
    a, b = g.download_state(), o.state()
    for k in b:
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), (what, k)


@pytest.mark.parametrize("kind,dim", [(1, 3), (3, 5)])
def test_single_calls_after_a_captured_setup(mdas, kind, dim):
    """A caller's graph that sets the grid up (InitialSampling, its integrand,
    ComputeErrors) is replayed after any number of passes: the host has not
    seen the tree start over, and the next single calls find it as it is."""
    from pmdas_amd import hip
    W, H = 48.0, 32.0
    args = (dim, 30000, 4, 0, 2, 0.25, W, H)
    g, sc = mdas.KDGrid(*args), mdas.Scene(kind, 5, dim, W, H)
    params = sc.params_bytes()
    st = hip.Stream()
    g.stream = st
    graph = hip.Graph(st)
    graph.begin()
    g.InitialSampling()
    g.EvalNewSamples(sc)
    g.ComputeErrors()
    graph.end()
    for turn in range(5):
        _say(f"captured setup {kind} replay {turn}")
        graph.launch()
        st.synchronize()
        o = pyoracle.OracleGrid(*args)
        o.initial_sampling()
        o.eval_scene(params, 0, o.n_samples)
        o.compute_errors()
        for p in range(1 + turn):  # odd and even numbers of passes
            if p == 0:
                g.AdaptiveSampling()
                o.adaptive_sampling()
            else:
                g.SamplingPass()
                o.sampling_pass()
            assert (g.GetNewSamples(), g.GetNewNodes()) == (o.new_samples, o.new_nodes)
            assert (g.GetNumberOfSamples(), g.GetNumberOfNodes()) == (o.n_samples, o.n_leaves)
            g.EvalNewSamples(sc)
            st.synchronize()
            o.eval_scene(params, o.n_samples - o.new_samples, o.new_samples)
            _check(g, o, (turn, p))
        o.close()
    g.stream = None
    graph.destroy()
    st.destroy()
    g.close()
    sc.close()


def test_max_error_brings_the_counts(mdas):
    """GetMaxError reads the grid's counters back, after which the host's
    counts are the tree's: also of one that a graph has started over."""
    from pmdas_amd import hip
    g, sc = mdas.KDGrid(3, 30000, 4, 0, 2, 0.25, 48.0, 32.0), mdas.Scene(1, 5, 3, 48.0, 32.0)
    st = hip.Stream()
    g.stream = st
    graph = hip.Graph(st)
    graph.begin()
    g.InitialSampling()
    graph.end()
    g.Run(sc, 3000)
    assert g.GetNumberOfSamples() >= 3000
    graph.launch()
    st.synchronize()
    assert g.GetMaxError() == 0.0
    assert (g.GetNumberOfSamples(), g.GetNumberOfNodes()) == (64, 16)
    assert (g.GetNewSamples(), g.GetNewNodes()) == (64, 0)
    g.Run(sc, 3000)
    n, e = g.GetNumberOfSamples(), g.GetMaxError()
    assert n == g.GetNumberOfSamples() >= 3000 and e > 0
    graph.destroy()
    st.destroy()
    g.close()
    sc.close()
