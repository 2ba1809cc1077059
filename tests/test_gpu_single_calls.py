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
