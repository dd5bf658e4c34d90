"""Host code of the library against a HIP runtime made of host memory
(fake_hip.cpp): what it allocates, launches and reports, without a GPU.  Each test
runs in a process of its own, in which the runtime's functions are loaded before
the library's."""

import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

HEAD = '''
import ctypes, sys
import numpy as np
sys.path[:0] = [{root!r}, {here!r}]
fake = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)
fake.fake_most_lds.restype = fake.fake_live_bytes.restype = ctypes.c_size_t
fake.fake_launches.restype = fake.fake_allocations.restype = ctypes.c_long
from gpu_models import plane_model, rich_model
from gprmax_amd.hip import HipBatch, HipSolver
from gprmax_amd.utilities import GeneralError
def add_pml(s, p):
    eR = np.ascontiguousarray(np.stack([p.ERA, p.ERB, p.ERE, p.ERF]), dtype=np.float32)
    hR = np.ascontiguousarray(np.stack([p.HRA, p.HRB, p.HRE, p.HRF]), dtype=np.float32)
    from gprmax_amd.pml import DIRECTION_CODE
    s._check(s.lib.gpx_add_pml(s.ctx, DIRECTION_CODE[p.direction], p.xs, p.xf, p.ys, p.yf, p.zs, p.zf, len(p.CFS),
                               float(p.d), eR.ctypes.data, hR.ctypes.data, None))
'''


@pytest.fixture(scope='module')
def runtime(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp('fake_hip') / 'libfake_hip.so')
    subprocess.run(['g++', '-std=c++17', '-O1', '-w', '-fPIC', '-shared', '-D__HIP_PLATFORM_AMD__', '-I/opt/rocm/include',
                    os.path.join(HERE, 'fake_hip.cpp'), '-o', lib], check=True)
    head = HEAD.format(root=os.path.dirname(HERE), here=HERE, lib=lib)

    def run(code):
        r = subprocess.run([sys.executable, '-c', head + textwrap.dedent(code)], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return run


def test_slabs_added_to_a_model_of_a_batch_get_their_phi(runtime):
    """A model that has its slabs when the batch is made, and one that gets them
    afterwards, hold the same arrays when the batch runs."""
    runtime('''
        for shape, pml in (((12, 13, 14), 3), ((12, 13, 14), {'x0': 3, 'zmax': 2})):
            G = [rich_model(seed=n, shape=shape, pml=pml, snapshots=False) for n in range(2)]
            for group in (0, 1):
                held = []
                for late in (False, True):
                    slabs = list(G[1].pmls)
                    G[1].pmls = [] if late else slabs
                    ss = [HipSolver(g) for g in G]
                    with HipBatch(ss) as b:
                        b.set_group_bytes(group)
                        for p in slabs if late else []:
                            add_pml(ss[1], p)
                        b.run(0, 4)
                        held.append(fake.fake_live_bytes())
                    for s in ss:
                        s.close()
                    G[1].pmls = slabs
                assert held[0] == held[1], held
    ''')


def test_an_allocation_that_fails_leaves_the_model_whole(runtime):
    """Every device allocation of a run fails once, on models that hold one or two
    states and on ones that get slabs between runs: the run reports it, and the
    next one holds what a model has whose allocations never failed."""
    runtime('''
        def models():
            yield rich_model(seed=1, shape=(12, 13, 14), pml=3, snapshots=False), 1
            yield rich_model(seed=2, shape=(12, 13, 14), pml=0, snapshots=False), 4
            yield plane_model(seed=3, axis=2, snapshots=False), 4
            yield rich_model(seed=4, shape=(12, 13, 14), poles=2, pml=3, snapshots=False), 4
        for G, form in models():
            slabs = list(G.pmls)
            for first in (slabs, slabs[:1], []):
                G.pmls = first
                def go(fail):
                    with HipSolver(G) as s:
                        s.set_step(form)
                        for phase in range(2):
                            if phase:
                                for p in slabs[len(first):]:
                                    add_pml(s, p)
                            fake.fake_fail_at(fail[phase])
                            if fail[phase]:
                                try:
                                    s.run(0, 3)
                                    raise SystemExit('no error')
                                except GeneralError as e:
                                    assert 'memory' in str(e), e
                            fake.fake_fail_at(0)
                            s.run(0, 3)
                            made[phase] = fake.fake_allocations()
                        return fake.fake_live_bytes()
                made = [0, 0]
                held, counts = go([0, 0]), list(made)
                assert counts[0] > 0
                for phase in range(2):
                    for n in range(1, counts[phase] + 1):
                        fail = [0, 0]
                        fail[phase] = n
                        assert go(fail) == held, (form, len(first), fail)
    ''')


@pytest.mark.parametrize('thick,rows', [(2000, True), (2100, False)])
def test_inversion_profiles_past_the_lds_take_the_general_kernels(thick, rows, runtime):
    """Slabs of 2 x 2100 cells have 67 KB of profile entries a field, more than the
    64 KB a block's tables may take; of 2 x 2000, 64 000 B."""
    runtime('''
        from gprmax_amd.inversion import InversionGeometry, InversionGrid
        init = InversionGeometry.__init__
        def only_x(self, *a, **k):
            init(self, *a, **k)
            self.slabs = [p for p in self.slabs if p.direction[0] == 'x']
        InversionGeometry.__init__ = only_x
        shape = ({n}, 8, 8)
        g = InversionGrid(shape, 2e-3, 2, pml={thick}, er_pml=6.0, K=1)
        g.set_model(np.full(shape, 6.0), np.zeros(shape))
        tr = g.forward(({n} // 2, 4, 4), [({n} // 2, 4, 5)], np.ones(2, np.float32))
        g.backward(tr)
        assert fake.fake_most_lds() <= 65536, fake.fake_most_lds()
        assert (fake.fake_launches(b'k_inv_row_h') > 0) is {rows}
        assert (fake.fake_launches(b'k_inv_h') > 0) is not {rows}
    '''.format(n=2 * thick + 20, thick=thick, rows=rows))


def test_an_allocation_that_fails_leaves_the_inversion_whole(runtime):
    """The same for the differentiable solver: poles set, a forward with other
    receivers, and a backward, which needs a forward that succeeded."""
    runtime('''
        from gprmax_amd.inversion import InversionGrid
        shape, w = (12, 13, 14), np.ones(6, np.float32)
        rx = [(5, 6, 7), (6, 6, 7)]
        debye = np.full((2,) + shape, 1.0), np.full((2,) + shape, 1e-10)
        base = fake.fake_live_bytes()
        def go(phase, n):
            g = InversionGrid(shape, 2e-3, 6, pml=3, er_pml=6.0, K=2)
            g.set_model(np.full(shape, 6.0), np.zeros(shape))
            g.set_keep(g.keep_bytes_all() / 3)
            def attempt(k, f):
                if k == phase and n:
                    fake.fake_fail_at(n)
                    try:
                        f()
                        raise SystemExit('no error')
                    except GeneralError as e:
                        assert 'memory' in str(e) or 'allocate' in str(e), e
                    fake.fake_fail_at(0)
                    try:
                        g.backward(np.zeros((2, 6)))
                        raise SystemExit('a backward without its forward')
                    except GeneralError as e:
                        assert 'gpx_inv_forward first' in str(e), e
                fake.fake_fail_at(0)
                f()
                if k == phase:
                    made[0] = fake.fake_allocations()
            attempt(0, lambda: g.forward((6, 6, 6), rx, w))
            attempt(1, lambda: g.set_debye(*debye))
            attempt(2, lambda: g.forward((6, 6, 6), rx, w))
            attempt(3, lambda: g.forward((6, 6, 6), rx[:1], w))
            g.backward(np.zeros((1, 6)))
            held = fake.fake_live_bytes()
            g.close()
            assert fake.fake_live_bytes() == base
            return held
        for phase in range(4):
            made = [0]
            held = go(phase, 0)
            counts = made[0]
            assert counts > 0
            for n in range(1, counts + 1):
                assert go(phase, n) == held, (phase, n)
    ''')


@pytest.mark.parametrize('poles', [0, 1])
def test_rows_of_two_points_are_not_padded(poles, runtime):
    """A TMz model holds what TMx and TMy models of its size hold, but for its Phi,
    whose rows of two are padded to eight."""
    runtime('''
        held = []
        for axis in range(3):
            with HipSolver(plane_model(seed=5, axis=axis, size=(399, 399), iterations=4, poles={poles}, snapshots=False)) as s:
                s.run(0, 4)
                held.append(fake.fake_live_bytes())
        assert max(held) < 1.1 * min(held), held
    '''.format(poles=poles))


@pytest.mark.parametrize('shape,poles,rows', [((620, 600, 500), 0, True), ((6000, 6000, 4), 1, False), ((620, 600, 440), 1, True)],
                         ids=str)
def test_states_past_4_gib_take_the_row_passes(shape, poles, rows, runtime):
    """187 million points without poles, 180 million with (their rows of five are
    then not padded to eight); 164 million are within 32-bit offsets."""
    runtime('''
        from types import SimpleNamespace
        shape, poles = {shape}, {poles}
        n = tuple(v + 1 for v in shape)
        table = np.ones((2, 5), np.float32)
        G = SimpleNamespace(nx=shape[0], ny=shape[1], nz=shape[2], iterations=30, floattype=np.float32, maxpoles=poles,
                            ID=np.zeros((6,) + n, np.uint32), updatecoeffsE=table, updatecoeffsH=table,
                            updatecoeffsdispersive=np.zeros((2, 3 * poles), np.complex64), pmlformulation='HORIPML', pmls=[],
                            hertziandipoles=[], magneticdipoles=[], voltagesources=[], transmissionlines=[], snapshots=[], rxs=[])
        with HipSolver(G) as s:
            s.set_step(6)
            s.run(0, 30)
            h, general = fake.fake_launches(b'k_row_h'), fake.fake_launches(b'k_h_pass')
            assert (h > 0, general > 0) == ({rows}, not {rows}), (h, general)
            points = float(np.prod(n))
            if poles and not {rows}:
                assert s.memory_bytes() < 50 * points, s.memory_bytes() / points
    '''.format(shape=shape, poles=poles, rows=rows))
