"""Edges of the differentiable solver's row kernels (csrc/inv_rows.h): row
lengths around the lanes' two cells, the padding and the wave, no slabs, poles,
receivers in the PML.  The gradient over every cell (the slabs' too) against
the float64 autograd reference, and against the general kernels, which run
the model when its slabs come in another order.

Tolerances: 1e-3 against float64, as in test_inversion.py; between the two
paths, which differ by the order in which a cell in two slabs adds their terms
(one rounding of 6e-8 an iteration, over 40 forward and 40 reverse ones, and a
gradient that sums over them), 1e-4.
"""

import numpy as np
import pytest
import torch

from gprmax_amd.inversion import InversionGeometry
from test_inversion import _autograd, _debye_params, _observed

pytestmark = pytest.mark.gpu


def _gradient(shape, pml, debye, args, monkeypatch, reverse):
    from gprmax_amd.inversion import InversionGrid, misfit_and_gradient
    init = InversionGeometry.__init__

    def reversed_init(self, *a, **k):
        init(self, *a, **k)
        self.slabs = self.slabs[::-1]
    if reverse:
        monkeypatch.setattr(InversionGeometry, '__init__', reversed_init)
    grid = InversionGrid(shape, 2e-3, 40, pml=pml, er_pml=7.0, K=16)
    monkeypatch.undo()
    try:
        if debye is not None:
            grid.set_debye(*debye)
        grid.interior = np.ones(shape, dtype=bool)
        return misfit_and_gradient(grid, *args)
    finally:
        grid.close()


@pytest.mark.parametrize('poles', [0, 2])
@pytest.mark.parametrize('shape,pml', [((13, 14, 15), 4), ((14, 13, 16), 4), ((12, 11, 17), 3), ((11, 12, 18), 3),
                                       ((10, 9, 131), 2), ((9, 10, 12), 0)], ids=str)
def test_gradient_at_the_edges_of_the_rows(shape, pml, poles, monkeypatch):
    rng = np.random.default_rng(60)
    geo = InversionGeometry(shape, 2e-3, 40, pml=pml, er_pml=7.0, K=16)
    debye = None
    if poles:
        debye = _debye_params(shape, 61, P=poles)
        geo.set_debye(*debye)
    waves = geo.waveform(freq=4e9)
    er_t, se_t = 4 + 6 * rng.random(shape), 1e-3 + 1.9e-2 * rng.random(shape)
    er0 = 7.0 + 0.3 * rng.standard_normal(shape)
    se0 = 1.05e-2 + 1e-3 * rng.standard_normal(shape)
    c = tuple(n // 2 for n in shape)
    src = [c]
    rx = [(c[0] - 1, c[1] + 1, c[2] + 1), (c[0] + 2, c[1], c[2] - 2), (1, 2, c[2] + 3)]
    obs = _observed(geo, waves, er_t, se_t, src, rx)
    L_ref, ger_ref, gse_ref = _autograd(geo, waves, er0, se0, src, rx, obs)
    args = (er0, se0, src, rx, obs, waves)
    L, ger, gse = _gradient(shape, pml, debye, args, monkeypatch, False)
    assert abs(L - L_ref) <= 1e-4 * L_ref
    m = geo.interior
    for ours, ref in ((ger, ger_ref), (gse, gse_ref)):
        assert np.linalg.norm((ours - ref)[m]) < 1e-3 * np.linalg.norm(ref[m])
    Lg, gerg, gseg = _gradient(shape, pml, debye, args, monkeypatch, True)
    assert abs(L - Lg) <= 1e-4 * Lg
    for ours, ref in ((ger, gerg), (gse, gseg)):
        assert np.linalg.norm(ours - ref) < 1e-4 * np.linalg.norm(ref)


@pytest.mark.parametrize('reverse', [False, True], ids=['rows', 'general'])
def test_many_receivers(reverse, monkeypatch):
    """300 receivers, several on a row and at a point, against one at a time: the
    same traces; a gradient against the float64 reference; and a forward of them
    takes no longer than three of one."""
    import time
    from gprmax_amd.inversion import InversionGrid
    shape, its = (40, 38, 39), 40
    rng = np.random.default_rng(62)
    init = InversionGeometry.__init__

    def reversed_init(self, *a, **k):
        init(self, *a, **k)
        self.slabs = self.slabs[::-1]
    if reverse:
        monkeypatch.setattr(InversionGeometry, '__init__', reversed_init)
    grid = InversionGrid(shape, 2e-3, its, pml=4, er_pml=7.0, K=16)
    monkeypatch.undo()
    geo = InversionGeometry(shape, 2e-3, its, pml=4, er_pml=7.0, K=16)
    waves = geo.waveform(freq=4e9)
    er, se = 4 + 6 * rng.random(shape), 1e-3 + 1.9e-2 * rng.random(shape)
    src = tuple(n // 2 for n in shape)
    rx = rng.integers(src[0] - 4, src[0] + 5, (300, 3))
    rx[:80, :2] = src[:2]
    rx[250:] = rx[200:250]
    grid.set_model(er, se)
    one = [grid.forward(src, rx[n:n + 1], waves)[0] for n in (0, 40, 79, 199, 225, 275, 299)]
    tr = grid.forward(src, rx, waves)
    for n, t in zip((0, 40, 79, 199, 225, 275, 299), one):
        assert np.array_equal(tr[n], t) and np.abs(t).max() > 0
    ger, gse = grid.backward(tr)
    _, ger_ref, gse_ref = _autograd(geo, waves, er, se, [src], [tuple(r) for r in rx], [np.zeros((300, its))])
    m = geo.interior
    for ours, ref in ((ger, ger_ref), (gse, gse_ref)):
        assert np.linalg.norm((ours - ref)[m]) < 1e-3 * np.linalg.norm(ref[m])

    def took(n):
        best = 1e9
        for _ in range(10):
            t = time.perf_counter()
            grid.forward(src, rx[:n], waves)
            best = min(best, time.perf_counter() - t)
        return best
    assert took(300) < 3 * took(1)
    grid.close()
