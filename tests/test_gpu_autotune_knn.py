"""The autotuner's kNN axis: wavefronts per workgroup are a shape of the heap's search only, so tuning the
search in registers leaves them as they were, and there they change no result."""
import numpy as np
import pytest

from skid_amd import skg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [32, 64])
@pytest.mark.parametrize("waves", [1, 2])
def test_search_in_registers_has_no_wave_axis(box1, k, waves, monkeypatch):
    monkeypatch.setenv("SKG_KNN_WAVES", str(waves))
    ctx = skg.Context(box1, skg.make_params(0.005, k, period=1.0))
    for _ in range(2):
        t = ctx.autotune(skg.SKG_TUNE_KNN)
        assert t["knn_bucket"] in (8, 16, 32, 64) and t["knn_waves"] == waves
    ctx.close()


@pytest.mark.parametrize("k", [31, 32, 33, 64])
def test_heap_search_by_one_or_two_wavefronts(box1, k, monkeypatch):
    got = []
    for waves in ("1", "2"):
        monkeypatch.setenv("SKG_KNN_WAVES", waves)
        ctx = skg.Context(box1, skg.make_params(0.005, k, period=1.0, accumulate=skg.SKG_ACC_PLAIN))
        b2, rho, _ = ctx.density()
        got.append((b2, rho, *ctx.neighbors()))
        ctx.close()
    for one, two in zip(*got):
        assert np.array_equal(one, two)
