"""Edges of the row kernels (csrc/gpx_rows.h) against the CPU oracle from a
random state: row lengths around the lanes' two cells and the rows' padding,
rows longer than a wave, slabs of one cell, slabs that meet or overlap (the
general passes), values of every magnitude down to the subnormal ones (the
slabs' division), materials with different H coefficients.

Both sides round every operation the same way, so the expected agreement is
bit for bit.
"""

import numpy as np
import pytest

import oracle
from oracle import solver as osolver
from gpu_models import plane_model, randomise_tables, rich_model
from test_gpu_parity import COMPS, _assert_state_equal, _hip, _push_state, _random_state

pytestmark = pytest.mark.gpu

FACES = {'x0': 3, 'y0': 2, 'z0': 4, 'xmax': 1, 'ymax': 4, 'zmax': 3}
MEET = {'x0': 4, 'y0': 4, 'z0': 4, 'xmax': 4, 'ymax': 4, 'zmax': 4}


def _check(G, form, xchunk, scale=None):
    _random_state(G, 9)
    if scale is not None:
        rng = np.random.default_rng(3)
        arrays = [getattr(G, c) for c in COMPS]
        for pml in G.pmls:
            arrays += [pml.EPhi1, pml.EPhi2, pml.HPhi1, pml.HPhi2]
        for a in arrays:
            a *= np.exp2(-rng.integers(0, scale, a.shape)).astype(np.float32)
    lib = oracle.load(np.float32)
    with _hip()(G) as s:
        s.set_step(form)
        s.set_launch(xchunk, 0)
        _push_state(s, G)
        s.run(0, 4)
        for it in range(4):
            osolver.step(lib, G, it, 8)
        _assert_state_equal(s, G, 'form {}'.format(form))


@pytest.mark.parametrize('form', [0, 1], ids=['passes', 'one-launch'])
@pytest.mark.parametrize('shape', [(13, 14, 12), (12, 15, 13), (14, 13, 14), (15, 12, 15), (12, 13, 127), (13, 12, 131)],
                         ids=str)
@pytest.mark.parametrize('order,formulation', [(1, 'HORIPML'), (2, 'HORIPML'), (1, 'MRIPML'), (2, 'MRIPML')])
def test_row_lengths(order, formulation, shape, form):
    G = rich_model(seed=50, shape=shape, iterations=8, snapshots=False, pml=FACES, order=order, formulation=formulation)
    _check(G, form, 3)


@pytest.mark.parametrize('block', [64, 512])
@pytest.mark.parametrize('shape', [(13, 14, 12), (12, 31, 33), (12, 13, 131)], ids=str)
@pytest.mark.parametrize('kind,poles', [('debye', 1), ('debye', 2), ('debye', 3), ('drude', 4), ('lorentz', 1), ('lorentz', 2),
                                        ('lorentz', 3), ('lorentz', 4)])
def test_auxiliary_values_by_groups(kind, poles, shape, block):
    """Slots from a wave's masks: planes that end within a group of lanes and
    blocks that end past the plane; edges with poles in one cell of a lane, in
    both, in none."""
    G = rich_model(seed=57, shape=shape, iterations=8, snapshots=False, pml=FACES, poles=poles, kind=kind)
    _random_state(G, 9)
    lib = oracle.load(np.float32)
    with _hip()(G) as s:
        s.set_launch(3, block)
        _push_state(s, G)
        s.run(0, 4)
        for it in range(4):
            osolver.step(lib, G, it, 8)
        _assert_state_equal(s, G, 'block {}'.format(block))


@pytest.mark.parametrize('tile', [256, 512, 1024])
@pytest.mark.parametrize('xchunk', [0, 1, 3])
@pytest.mark.parametrize('pml', [0, FACES], ids=['open', 'slabs'])
def test_dipoles_on_recomputed_cells(pml, xchunk, tile):
    """The one-launch step computes H of a tile's halo again: the row below it, the
    lane before it where rows are split, the plane before each chunk.  Magnetic
    dipoles along whole lines of every axis, which cross all of these, are in the
    copies as in the owners' values."""
    from gprmax_amd.grid import ModelBuilder
    shape = (11, 29, 141)

    def model():
        bld = ModelBuilder(*shape, 1e-3, 1e-3, 1e-3, 9, pml_cells=pml)
        soil = bld.add_material(4.0, 0.005, 1, 0, 'soil')
        bld.box(0, shape[0], 0, shape[1], 0, shape[2] // 2, soil)
        bld.add_waveform('ricker', 1, 20e9, 'w')
        lo, hi = (5, 5, 5), tuple(n - 5 for n in shape)
        for pol, a in zip('xyzxyz', (0, 1, 2, 1, 2, 0)):
            for c in range(lo[a], hi[a]):
                at = [lo[0] + 1, lo[1] + 3, lo[2] + 40]
                at[a] = c
                bld.add_magnetic_dipole(pol, tuple(at), 'w')
        bld.add_hertzian_dipole('z', tuple(n // 2 for n in shape), 'w')
        for k in (6, 61, 63, 64, 65, 127, 129):
            bld.add_rx((6, 8, k))
        return bld.finalise()
    G, Gc = model(), model()
    with _hip()(G) as s:
        s.set_step(1, tile)
        s.set_launch(xchunk, 0)
        assert s.step_kind() == tile
        s.run(0, G.iterations)
        F, rxb = s.download_fields(), s.download_rx()
    osolver.solve_cpu(1, 1, Gc, nthreads=8)
    for n, c in enumerate(COMPS):
        assert np.abs(F[n]).max() > 0 and np.array_equal(F[n], getattr(Gc, c)), c
    for r, rx in enumerate(Gc.rxs):
        for c, name in enumerate(COMPS):
            assert np.array_equal(rxb[c, :, r], rx.outputs[name]), (r, name)


@pytest.mark.parametrize('form', [0, 1], ids=['passes', 'one-launch'])
@pytest.mark.parametrize('magnetic', [False, True])
def test_values_of_every_magnitude(magnetic, form):
    G = rich_model(seed=51, shape=(13, 14, 15), iterations=8, snapshots=False, pml=FACES)
    if magnetic:
        randomise_tables(G, 52, scaled=True)
    _check(G, form, 0, scale=145)


@pytest.mark.parametrize('form', [0, 1], ids=['passes', 'one-launch'])
@pytest.mark.parametrize('cell', [0, 1])
def test_tiny_values_in_one_cell_of_a_lane(cell, form):
    """Fields of 2^-126 to 2^-148 in one of a lane's two cells and zero in the
    other: the slabs' quotient of either cell is that of the division."""
    G = rich_model(seed=52, shape=(13, 14, 15), iterations=8, snapshots=False, pml=FACES)
    _random_state(G, 9)
    for c in COMPS:
        a = getattr(G, c)
        a *= np.exp2(-np.random.default_rng(4).integers(126, 149, a.shape).astype(np.float32))
        a[:, :, 1 - cell::2] = 0
    for pml in G.pmls:
        for a in (pml.EPhi1, pml.EPhi2, pml.HPhi1, pml.HPhi2):
            a[:] = 0
    lib = oracle.load(np.float32)
    with _hip()(G) as s:
        s.set_step(form)
        _push_state(s, G)
        s.run(0, 1)
        osolver.step(lib, G, 0, 8)
        _assert_state_equal(s, G, 'form {}'.format(form))


@pytest.mark.parametrize('form', [0, 1], ids=['passes', 'one-launch'])
@pytest.mark.parametrize('value', [np.inf, -np.inf, np.nan, 3e38, -2e36], ids=str)
def test_quotients_that_overflow(value, form):
    """Fields with a few infinities, or values whose quotient by the cell size
    overflows, in either cell of a lane: infinities and NaN are where the
    division leaves them."""
    G = rich_model(seed=58, shape=(13, 14, 15), iterations=8, snapshots=False, pml=FACES)
    _random_state(G, 9)
    rng = np.random.default_rng(5)
    for c in COMPS:
        a = getattr(G, c)
        a[rng.random(a.shape) < 0.02] = value
    lib = oracle.load(np.float32)
    with _hip()(G) as s:
        s.set_step(form)
        _push_state(s, G)
        s.run(0, 1)
        osolver.step(lib, G, 0, 8)
        F = s.download_fields()
        for n, c in enumerate(COMPS):
            assert np.array_equal(F[n], getattr(G, c), equal_nan=True), c
        for n, pml in enumerate(G.pmls):
            for w, name in enumerate(('EPhi1', 'EPhi2', 'HPhi1', 'HPhi2')):
                assert np.array_equal(s.download_phi(n, w), getattr(pml, name), equal_nan=True), (pml.ID, name)
        assert np.isinf(F).any() or np.isnan(value)


@pytest.mark.parametrize('axis', [0, 1, 2], ids=['TMx', 'TMy', 'TMz'])
def test_2d_quotients_that_overflow(axis):
    """The same for the 2-D kernel, from sources in and beside the slabs, against
    the general passes."""
    G = plane_model(seed=63, axis=axis, size=(25, 24), iterations=30, snapshots=False)
    cells = np.zeros((6, 6), np.int32)
    u, v = (a for a in range(3) if a != axis)
    cells[:, u], cells[:, v] = (1, 2, 5, 12, 21, 23), (12, 3, 20, 4, 9, 21)
    cells[:, 3], cells[:, 5] = axis, 29
    fac, waves = np.ones((6, 2), np.float32), np.zeros((6, 30), np.float32)
    waves[:, 3] = (3e38, -3e38, 1e36, np.inf, -1e37, 2e38)
    got = []
    for form in (4, 2):
        with _hip()(G) as s:
            s.set_step(form)
            s._check(s.lib.gpx_set_sources(s.ctx, 0, 6, cells.ctypes.data, fac.ctypes.data, waves.ctypes.data))
            s.run(0, 5)
            got.append(s.download_fields())
    assert np.isinf(got[0]).any()
    assert np.array_equal(got[0], got[1], equal_nan=True)


@pytest.mark.parametrize('form', [0, 1], ids=['passes', 'one-launch'])
@pytest.mark.parametrize('shape', [(10, 12, 12), (12, 10, 12), (12, 12, 9), (12, 12, 10)], ids=str)
def test_slabs_close_to_the_opposite_one(shape, form):
    G = rich_model(seed=53, shape=shape, iterations=8, snapshots=False, pml=MEET)
    _check(G, form, 0)


def test_indices_of_several_pieces_are_checked_to_the_last():
    """129 x 119 x 181 points x 6 indices are two pieces of the upload; an
    index past the tables is refused wherever it is, the first one named, and
    the model then takes good indices and keeps them when more bad ones come."""
    from gprmax_amd.grid import ModelBuilder
    from gprmax_amd.utilities import GeneralError
    G = ModelBuilder(128, 118, 180, 1e-3, 1e-3, 1e-3, 4, pml_cells=4).finalise()
    good = G.ID.copy()
    for at in ((0, 0, 0, 0), (2, 64, 7, 180), (5, 128, 118, 180)):
        G.ID = good.copy()
        G.ID[at] = 60000 + at[0]
        G.ID[5, 128, 118, 180] = max(60001, G.ID[5, 128, 118, 180])
        with pytest.raises(GeneralError, match='material index {} '.format(G.ID[at])):
            _hip()(G)
    G.ID = good
    with _hip()(G) as s:
        bad = good.copy()
        bad[3, 2, 1, 0] = 70000
        with pytest.raises(GeneralError, match='material index 70000 '):
            s._check(s.lib.gpx_upload_id(s.ctx, np.ascontiguousarray(bad, dtype=np.uint32).ctypes.data))
        s.run(0, 4)
        assert not np.any(s.download_fields())


@pytest.mark.parametrize('shape,poles,magnetic', [((60, 380, 362), 0, False), ((61, 330, 300), 2, True), ((12, 870, 701), 0, True)],
                         ids=str)
def test_blocks_of_planes(shape, poles, magnetic):
    """Grids past the last-level cache go through the passes in blocks of planes
    that move with the iterations, fewer planes than iterations too; sources,
    receivers, snapshots between and runs of one iteration: as whole general
    passes give it, bit for bit."""
    G = rich_model(seed=54, shape=shape, iterations=40, pml=FACES, poles=poles)
    if magnetic:
        randomise_tables(G, 55, scaled=True)
    for n, s in enumerate(G.snapshots):
        s.time = 5 + 14 * n
    rng = np.random.default_rng(56)
    F = rng.standard_normal((6,) + tuple(n + 1 for n in shape), dtype=np.float32)
    got = []
    for form in (4, 2):
        with _hip()(G) as s:
            s.set_step(form)
            s.upload_fields(F)
            for it, n in ((0, 23), (23, 1), (24, 2), (26, 9)):
                s.run(it, n)
            got.append([s.download_fields(), s.download_rx()] + [s.download_phi(p, w) for p in range(6) for w in range(4)]
                       + [s.download_snapshot(n) for n in range(len(G.snapshots))] + ([s.download_T()] if poles else []))
    for n, (a, b) in enumerate(zip(*got)):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), n


@pytest.mark.parametrize('order,formulation,uniform', [(0, 'HORIPML', True), (1, 'HORIPML', True), (2, 'HORIPML', False),
                                                       (1, 'MRIPML', False), (2, 'MRIPML', True)])
def test_states_past_4_gib(order, formulation, uniform):
    """180 million points, whose state 32-bit offsets do not reach across: sources,
    receivers and slabs at the far end of every component, as whole general
    passes give it, bit for bit."""
    from types import SimpleNamespace
    shape = (700, 640, 401)
    n = tuple(v + 1 for v in shape)
    points = n[0] * n[1] * n[2]
    assert points * 24 > 2 ** 32
    G = rich_model(seed=66, shape=(24, 23, 22), iterations=40, order=max(order, 1), formulation=formulation,
                   pml={'xmax': 4, 'ymax': 3, 'zmax': 4} if order else 0, snapshots=False)
    if not uniform:
        randomise_tables(G, 67, scaled=True)
    nmat = len(G.updatecoeffsE)
    pattern = np.random.default_rng(68).integers(0, nmat, 999983, dtype=np.uint32)
    move = [a - b for a, b in zip(shape, (24, 23, 22))]
    slabs = []
    for p in G.pmls:    # the faces at the far end, as thick as they were
        q = SimpleNamespace(**{k: getattr(p, k) for k in ('direction', 'd', 'CFS', 'ERA', 'ERB', 'ERE', 'ERF', 'HRA', 'HRB', 'HRE', 'HRF')})
        a = 'xyz'.index(p.direction[0])
        for x, name in enumerate('xyz'):
            lo, hi = getattr(p, name + 's'), getattr(p, name + 'f')
            setattr(q, name + 's', lo + move[x] if x == a else 0)
            setattr(q, name + 'f', hi + move[x] if x == a else shape[x])
        slabs.append(q)
    big = SimpleNamespace(**{k: getattr(G, k) for k in ('iterations', 'updatecoeffsE', 'updatecoeffsH', 'pmlformulation', 'dx', 'dy',
                                                        'dz', 'dt')},
                          nx=shape[0], ny=shape[1], nz=shape[2], floattype=np.float32, maxpoles=0, pmls=slabs,
                          ID=np.resize(pattern, (6,) + n), hertziandipoles=[], magneticdipoles=[], voltagesources=[],
                          transmissionlines=[], snapshots=[],
                          rxs=[SimpleNamespace(xcoord=r.xcoord + move[0], ycoord=r.ycoord + move[1], zcoord=r.zcoord + move[2])
                               for r in G.rxs])
    F = np.empty((6,) + n, np.float32)
    got = []
    for form in (4, 2):
        with _hip()(big) as s:
            s.set_step(form)
            for kind, pol in ((0, 2), (1, 1), (2, 0)):
                at = np.array([[700 - 9, 640 - 8, 401 - 9, pol, 0, 39], [12, 11, 10, pol, 0, 39]], np.int32)
                fac, waves = np.full((2, 2), 2.0, np.float32), np.random.default_rng(69).random((2, 40), dtype=np.float32)
                s._check(s.lib.gpx_set_sources(s.ctx, kind, 2, at.ctypes.data, fac.ctypes.data, waves.ctypes.data))
            s.run(0, 27)
            s._check(s.lib.gpx_download_fields(s.ctx, F.ctypes.data))
            got.append([F[:, -60:, -60:, -60:].copy(), F[:, :60, :60, :60].copy(), s.download_rx()])
            if form == 4:
                F[:, -60:, -60:, -60:] = 0
                F[:, :60, :60, :60] = 0
                assert not F.any()
    for a, b in zip(*got):
        assert np.abs(a).max() > 0 and np.array_equal(a, b)


@pytest.mark.parametrize('n', [1, 7, 31], ids=['n1', 'n7', 'n31'])
@pytest.mark.parametrize('size', [(14, 17), (25, 24), (57, 90), (300, 211)], ids=str)
@pytest.mark.parametrize('axis', [0, 1, 2], ids=['TMx', 'TMy', 'TMz'])
def test_2d_tiles(axis, size, n):
    """Several iterations of a 2-D model in one launch, planes smaller and
    larger than a tile, sources on one edge and several receivers at one point,
    between snapshots and in stretches of n; as the passes give it, bit for bit."""
    G = plane_model(seed=60 + n, axis=axis, size=size, iterations=62, order=1 + n % 2,
                    formulation='MRIPML' if n == 7 else 'HORIPML')
    G.rxs = G.rxs + G.rxs[:1] + G.rxs[-1:]
    G.hertziandipoles = G.hertziandipoles + G.hertziandipoles[:1]
    got = []
    for form in (4, 6):
        with _hip()(G) as s:
            s.set_step(form)
            for it in range(0, 62, n):
                s.run(it, min(n, 62 - it))
            got.append([s.download_fields(), s.download_rx(), s.download_snapshot(0)]
                       + [s.download_phi(p, w) for p in range(len(G.pmls)) for w in range(4)])
    assert np.abs(got[0][0]).max() > 0
    for q, (a, b) in enumerate(zip(*got)):
        assert np.array_equal(a, b), q
    # what the tiles' kernel leaves out may not be zero: the passes run
    F = np.random.default_rng(61).standard_normal(got[0][0].shape).astype(np.float32)
    out = []
    for form in (4, 6):
        with _hip()(G) as s:
            s.set_step(form)
            s.run(0, 9)
            s.upload_fields(F)
            s.run(9, 3)
            out.append(s.download_fields())
    assert np.array_equal(*out)


@pytest.mark.parametrize('order', [1, 2])
def test_states_of_several_pieces(order):
    """Fields and Phi larger than a piece of their transfers, rows with and without
    padding: what went up comes down, and one iteration from it is that of
    whole general passes."""
    from gprmax_amd.grid import ModelBuilder
    from gprmax_amd.pml import CFS
    cfs = [CFS() for _ in range(order)]
    for nz in (62, 63):
        b = ModelBuilder(220, 170, nz, 1e-3, 1e-3, 1e-3, 4, pml_cells={'x0': 29, 'zmax': 25}, cfs=cfs)
        G = b.finalise()
        rng = np.random.default_rng(65)
        F = rng.standard_normal((6, 221, 171, nz + 1), dtype=np.float32)
        out = []
        for form in (4, 2):
            with _hip()(G) as s:
                s.set_step(form)
                s.run(0, 1)
                P = {(p, w): rng.standard_normal(s.download_phi(p, w).shape, dtype=np.float32) for p in range(2) for w in range(4)}
                if out:
                    P = phi
                phi = P
                s.upload_fields(F)
                for k, v in P.items():
                    s.upload_phi(*k, v)
                assert np.array_equal(s.download_fields(), F)
                for k, v in P.items():
                    assert np.array_equal(s.download_phi(*k), v), k
                s.run(1, 2)
                out.append([s.download_fields()] + [s.download_phi(*k) for k in P])
        for a, c in zip(*out):
            assert np.array_equal(a, c)


def test_padded_rows_transfer_as_fast_as_whole_ones():
    """Rows of 182 points, padded on the device, against rows of 184: the fields
    take at most twice as long either way."""
    import time
    from gprmax_amd.grid import ModelBuilder
    took = []
    for nz in (181, 183):
        G = ModelBuilder(90, 90, nz, 1e-3, 1e-3, 1e-3, 4, pml_cells=4).finalise()
        with _hip()(G) as s:
            F = s.download_fields()
            down = up = 1e9
            for _ in range(8):
                t = time.perf_counter()
                s._check(s.lib.gpx_download_fields(s.ctx, F.ctypes.data))
                u = time.perf_counter()
                s._check(s.lib.gpx_upload_fields(s.ctx, F.ctypes.data))
                down, up = min(down, u - t), min(up, time.perf_counter() - u)
            took.append((down, up))
    assert took[0][0] < 2 * took[1][0] and took[0][1] < 2 * took[1][1], took


def test_2d_source_of_another_component_stays_in_the_state():
    """A 2-D run with a source off the plane's components, then without it: the
    later run goes on from what the source left, as the passes do."""
    import ctypes
    G = plane_model(seed=62, axis=2, size=(40, 33), iterations=40, snapshots=False)
    out = []
    for form in (4, 6):
        with _hip()(G) as s:
            s.set_step(form)
            info = np.array([[5, 16, 0, 2, 0, 39], [20, 16, 0, 2, 0, 39]], np.int32)        # along z
            fac, waves = np.full((2, 2), 3.0, np.float32), np.ones((2, 40), np.float32)
            ptr = [a.ctypes.data_as(ctypes.c_void_p) for a in (info, fac, waves)]
            s._check(s.lib.gpx_set_sources(s.ctx, 1, 2, *ptr))
            s.run(0, 11)
            s._check(s.lib.gpx_set_sources(s.ctx, 1, 0, None, None, None))
            s.run(11, 20)
            out.append(s.download_fields())
    assert np.abs(out[0][2]).max() > 0 and np.abs(out[0][5]).max() > 0
    assert np.array_equal(*out)


@pytest.mark.parametrize('group_bytes', [0, 1], ids=['one-group', 'each-alone'])
def test_slabs_added_after_the_batch_was_made(group_bytes):
    """A model of a batch that gets its slabs after the batch was made, between
    runs of it too, ends as one that is run alone."""
    from gprmax_amd.hip import HipBatch
    from gprmax_amd.pml import DIRECTION_CODE
    models = [rich_model(seed=64 + n, shape=(14, 13, 15), iterations=12, snapshots=False, pml=3) for n in range(2)]

    def add(s, p):
        R = [np.ascontiguousarray(np.stack([getattr(p, f + q) for q in ('RA', 'RB', 'RE', 'RF')]), np.float32) for f in 'EH']
        s._check(s.lib.gpx_add_pml(s.ctx, DIRECTION_CODE[p.direction], p.xs, p.xf, p.ys, p.yf, p.zs, p.zf, len(p.CFS),
                                   float(p.d), R[0].ctypes.data, R[1].ctypes.data, None))
    slabs = models[1].pmls
    out = []
    for batch in (False, True):
        models[1].pmls = []
        ss = [_hip()(G) for G in models]
        models[1].pmls = slabs
        b = HipBatch(ss) if batch else None
        if batch:
            b.set_group_bytes(group_bytes)
        for first, n, new in ((0, 5, slabs[:2]), (5, 7, slabs[2:])):
            for p in new:
                add(ss[1], p)
            if batch:
                b.run(first, n)
            else:
                for s in ss:
                    s.run(first, n)
        out.append([(s.download_fields(), s.download_rx()) for s in ss]
                   + [[ss[1].download_phi(p, w) for p in range(6) for w in range(4)]])
        if batch:
            b.close()
        for s in ss:
            s.close()
    for a, c in zip(*out):
        for x, y in zip(a, c):
            assert np.abs(x).max() > 0 and np.array_equal(x, y)
