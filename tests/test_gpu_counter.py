"""The device counter of replayed iterations over many runs: it follows by
itself from run to run, is set again where the draws jump or its history is
full, and its status word is clean after a run that reported NaN."""
import warnings

import numpy as np
import pytest
import torch

import vegasflow_amd as vf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cls,kwargs", [(vf.VegasFlow, {}), (vf.PlainFlow, {}), (vf.VegasFlowPlus, {"adaptive": True})])
def test_counter_follows_many_runs(cls, kwargs):
    """Thirteen runs of seven iterations (past the 64 history slots), with a
    sampling call, a new seed and a run on another stream between them,
    against the eager loop: every iteration to summation order (1e-10 over
    the refinements)."""
    pair = []
    for graphs in (False, True):
        inst = cls(3, 20_000, seed=3, verbose=False, **kwargs)
        inst.use_graphs = graphs
        inst.compile(vf.Gaussian(0.2, 0.4))
        for run in range(13):
            if run == 4:
                inst.generate_random_array(inst.n_events)  # takes a draw
            if run == 8:
                inst.set_seed(77)
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side if run == 10 else torch.cuda.current_stream()):
                inst.run_integration(7)
        pair.append(inst)
    eager, replayed = pair
    assert replayed._counter.capacity < 13 * 7
    assert len(eager.history) == len(replayed.history) == 13 * 7
    for (ra, ea, _), (rb, eb, _) in zip(eager.history, replayed.history):
        assert abs(ra - rb) <= 1e-10 * abs(ra) and abs(ea - eb) <= 1e-8 * abs(ea)
    assert eager._draw_count == replayed._draw_count
    if cls is vf.VegasFlowPlus:
        assert eager.events_history == replayed.events_history and eager.n_events == replayed.n_events


def test_status_is_clean_after_a_nonfinite_run():
    inst = vf.VegasFlow(2, 10_000, seed=5, verbose=False)
    inst.compile(vf.Constant(float("nan")))
    with pytest.warns(RuntimeWarning):
        inst.run_integration(3)
    assert inst.nonfinite_iterations == [0, 1, 2]
    inst.compile(vf.Gaussian(0.2, 0.4))
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        res, sigma = inst.run_integration(3)
    assert inst.nonfinite_iterations == [] and np.isfinite(res) and sigma > 0.0


def test_averages_with_zero_sigma_keep_the_array_arithmetic():
    """sigma = 0 (weights of infinity): NaN from inf / inf as before, no
    exception."""
    from vegasflow_amd.monte_carlo import _scalar_average

    assert _scalar_average([(np.float64(1.0), np.float64(0.0))]) is None
    r, s, chi2 = _scalar_average([(np.float64(1.0), np.float64(0.5)), (np.float64(2.0), np.float64(0.25))])
    w = np.array([4.0, 16.0])
    assert r == (1.0 * 4.0 + 2.0 * 16.0) / 20.0 and s == np.sqrt(1.0 / 20.0)
    assert abs(chi2 - np.sum(w * (np.array([1.0, 2.0]) - r) ** 2)) < 1e-14
