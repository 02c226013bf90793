"""CPU: the TL comparison of the GPU tests rejects fields that lack energy."""
import numpy as np
import pytest

from parity import tl_err


def _field():
    rng = np.random.default_rng(0)
    return (1e-4 * (rng.normal(size=(1, 30, 40)) + 1j * rng.normal(size=(1, 30, 40)))).astype(np.complex64)


def test_equal_and_scaled_fields():
    f = _field()
    assert tl_err(f, f) == 0.0
    assert tl_err(f * np.float32(1.01), f) == pytest.approx(20 * np.log10(1.01), rel=1e-3)


@pytest.mark.parametrize("part", [np.s_[:], np.s_[:, :20], np.s_[:, :, 3], np.s_[:, 29:, 39:]])
def test_missing_energy_is_an_error_either_way(part):
    f = _field()
    g = f.copy()
    g[part] = 0
    assert tl_err(g, f) > 100 and tl_err(f, g) > 100


def test_nothing_to_compare_is_an_error():
    assert tl_err(np.zeros((1, 2, 2)), np.zeros((1, 2, 2))) == np.inf
