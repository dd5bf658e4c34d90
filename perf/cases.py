"""Timed cases of the solver: what a modelling program has it do.

Four kinds of work, each through the package's public entry points:

* ``solve``: one whole model, host arrays to receiver traces and snapshots
  (``solve_hip``, the call that replaces the GPU solve of a model run);
* ``steps``: a model that is resident on the device advances by a stretch of
  iterations and its receivers and snapshot are read (``HipSolver``), as a
  program does that watches or steers a long run;
* ``bscan``: the traces of a B-scan, every trace its own domain
  (``solve_bscan``);
* ``gradient``: one source of a permittivity and conductivity inversion:
  forward traces, residual, gradient (``InversionGrid``).

Models are the ones of the package's workloads, tests and benchmark at their
sizes or other sizes of the same kind: free space, soil of random
non-dispersive materials under air, soil with Debye, Lorentz or Drude
materials, 2-D planes; HORIPML and MRIPML of one or two terms.
"""

import numpy as np
import torch

from gprmax_amd.grid import ModelBuilder
from gprmax_amd.hip import HipSolver, solve_bscan
from gprmax_amd.inversion import InversionGrid
from gprmax_amd.materials import add_dispersion
from gprmax_amd.pml import CFS
from gprmax_amd.solver import solve_hip


def _model(kind, nx, ny, nz, its, ground='soil', poles=0, nmat=64, share=1.0, pml=10, form='HORIPML', order=1,
           source='hertzian', cell=2e-3, name=None):
    c = {'kind': kind, 'nx': nx, 'ny': ny, 'nz': nz, 'its': its, 'ground': ground, 'poles': poles, 'nmat': nmat,
         'share': share, 'pml': pml, 'form': form, 'order': order, 'source': source, 'cell': cell}
    if name:
        c['name'] = name
    return c


def listed():
    return [
        # the 2-D A-scan every beginner runs: a TMz plane of 120 x 105 cells
        # over 3 ns; all launches and latency
        _model('solve', 120, 105, 1, 637, ground='box', name='ascan_2d_120x105'),
        # the basic 3-D test model: a dipole in free space, 100^3, 500 steps
        _model('solve', 100, 100, 100, 500, ground='free', cell=1e-3, name='freespace_100'),
        # an ordinary model with the other PML formulation, two CFS terms and
        # a voltage source, ragged sides
        _model('steps', 157, 131, 97, 150, pml=8, form='MRIPML', order=2, source='voltage', name='mripml2_157x131x97'),
        # the heterogeneous half-space at its full size, resident
        _model('steps', 300, 300, 200, 100, nmat=256, source='magnetic', name='halfspace_300x300x200'),
        # the same as one whole model run, set-up and read-out included
        _model('solve', 300, 300, 200, 600, nmat=256, source='magnetic', name='halfspace_solve'),
        # a thin, wide survey area: odd sides, short columns
        _model('steps', 611, 407, 45, 80, nmat=16, name='survey_611x407x45'),
        # three-pole Debye soil, 30 % of the cells dispersive, 20-cell PML
        _model('steps', 240, 240, 180, 50, ground='debye', poles=3, nmat=256, share=0.3, pml=20,
               name='debye3_240x240x180'),
        # a Lorentz medium filling the ground: complex auxiliary values
        _model('steps', 121, 104, 90, 120, ground='lorentz', poles=2, nmat=9, name='lorentz2_121x104x90'),
        # a B-scan of small uneven traces, several to the device at a time
        {'kind': 'bscan', 'traces': 10, 'lo': 56, 'hi': 96, 'its': 300, 'name': 'bscan_10_small'},
        # uneven traces of 128-256 cells a side
        {'kind': 'bscan', 'traces': 4, 'lo': 128, 'hi': 256, 'its': 300, 'name': 'bscan_4_uneven'},
        # a small inversion model with three Debye poles per cell
        {'kind': 'gradient', 'nx': 40, 'ny': 40, 'nz': 40, 'its': 150, 'K': 64, 'poles': 3, 'name': 'gradient_debye_40'},
        # one source of the full-size inversion
        {'kind': 'gradient', 'nx': 160, 'ny': 160, 'nz': 120, 'its': 600, 'K': 64, 'poles': 0,
         'name': 'gradient_160x160x120'},
    ]


def _sides(rng, lo, hi):
    """Three sides whose product is spread evenly over the logarithm of
    [lo, hi] cells, at most a factor of about four apart."""
    n = 2.718281828459045 ** rng.uniform(np.log(lo), np.log(hi))
    f = [2.0 ** rng.uniform(-1, 1) for _ in range(3)]
    g = (n / (f[0] * f[1] * f[2])) ** (1.0 / 3.0)
    return [max(26, int(round(g * v))) for v in f]


def draw(rng):
    kind = rng.choice(['steps', 'steps', 'steps', 'steps', 'solve', 'solve', 'bscan', 'gradient'])
    if kind == 'bscan':
        lo, hi = rng.choice([(48, 80), (64, 110), (90, 160), (128, 230)])
        traces = rng.randint(3, 9) if lo < 90 else rng.randint(2, 4)
        return {'kind': kind, 'traces': traces, 'lo': lo, 'hi': hi, 'its': rng.randint(120, 300)}
    if kind == 'gradient':
        nx, ny, nz = _sides(rng, 40000, 2500000)
        return {'kind': kind, 'nx': nx, 'ny': ny, 'nz': nz, 'its': rng.randint(90, 320), 'K': rng.choice([32, 50, 64]),
                'poles': rng.choice([0, 0, 0, 1, 3])}
    ground = rng.choice(['free', 'soil', 'soil', 'soil', 'box', 'debye', 'lorentz', 'drude'])
    poles = {'debye': rng.choice([1, 2, 3]), 'lorentz': rng.choice([1, 2]), 'drude': 1}.get(ground, 0)
    if rng.random() < 0.12:  # a 2-D plane
        sides = [rng.randint(60, 500), rng.randint(60, 500), 1]
        rng.shuffle(sides)
        nx, ny, nz = sides
        ground = 'soil' if ground == 'box' else ground
    else:
        nx, ny, nz = _sides(rng, 60000, 16000000 if not poles else 9000000)
    its = rng.randint(40, 160) if kind == 'steps' else rng.randint(120, 400)
    return _model(kind, nx, ny, nz, its, ground=ground, poles=poles, nmat=rng.choice([5, 16, 64, 200, 256]),
                  share=rng.choice([0.1, 0.3, 1.0]) if poles else 1.0, pml=rng.choice([5, 8, 10, 10, 10, 12]),
                  form=rng.choice(['HORIPML', 'HORIPML', 'HORIPML', 'MRIPML']), order=rng.choice([1, 1, 1, 2]),
                  source=rng.choice(['hertzian', 'hertzian', 'magnetic', 'voltage']), cell=rng.choice([1e-3, 2e-3]))


# ------------------------------------------------------------------ inputs
def _materials(b, rng, count, lossy=True):
    er, se = rng.uniform(3, 15, count), rng.uniform(1e-3, 5e-2, count) if lossy else np.zeros(count)
    return [b.add_material(float(er[n]), float(se[n]), 1, 0, 'm{}'.format(n)) for n in range(count)]


def _grid(case, seed):
    """The built grid of a `solve` or `steps` case: what the solver is given."""
    rng = np.random.default_rng(seed)
    nx, ny, nz, d = case['nx'], case['ny'], case['nz'], case['cell']
    cfs = None
    if case['order'] == 2:
        one, two = CFS(), CFS()
        one.alpha.max = 0.05
        two.kappa.scalingprofile, two.kappa.min, two.kappa.max = 'quadratic', 1, 3
        cfs = [one, two]
    b = ModelBuilder(nx, ny, nz, d, d, d, case['its'], pml_cells=case['pml'], pml_formulation=case['form'], cfs=cfs)
    flat = [n for n, v in enumerate((nx, ny, nz)) if v == 1]  # the invariant axis of a 2-D plane
    up = max(n for n in range(3) if n not in flat)
    size = (nx, ny, nz)
    ground = [slice(0, n) for n in size]
    if not case['poles']:
        ground[up] = slice(0, size[up] // 2)
    ground = tuple(ground)
    if case['ground'] == 'box':  # one averaged half-space
        m = b.add_material(float(rng.uniform(4, 9)), 0, 1, 0, 'half_space')
        b.box(*(v for s in ground for v in (s.start, s.stop)), m, averaging=True)
    elif case['ground'] != 'free':
        mats = _materials(b, rng, case['nmat'])
        first, n = mats[0].numID, len(mats)
        disp = mats[:max(1, n // 4)] if case['share'] < 1 else mats
        for m in disp if case['poles'] else []:
            p = case['poles']
            if case['ground'] == 'debye':
                add_dispersion(m, 'debye', list(rng.uniform(0.5, 5, p)), list(10 ** rng.uniform(-11, -8, p)))
            elif case['ground'] == 'lorentz':
                add_dispersion(m, 'lorentz', list(rng.uniform(0.5, 5, p)), list(rng.uniform(1e9, 5e9, p)),
                               list(rng.uniform(1e8, 5e8, p)))
            else:
                add_dispersion(m, 'drude', None, list(rng.uniform(1e9, 3e9, p)), list(rng.uniform(1e9, 5e9, p)))
        mask = np.zeros(size, dtype=bool)
        mask[ground] = True
        shape = mask[ground].shape
        ids = np.ones(size, dtype=np.uint32)
        if case['poles'] and case['share'] < 1:
            some = rng.random(shape) < case['share']
            ids[ground] = np.where(some, rng.integers(first, first + len(disp), shape),
                                   rng.integers(first + len(disp) if n > 1 else first, first + n, shape))
        else:
            ids[ground] = rng.integers(first, first + n, shape, dtype=np.uint32)
        b.paint_voxels(mask, ids)
    b.add_waveform('ricker', float(rng.uniform(0.5, 2)), float(rng.uniform(1.0e9, 2.0e9)), 'w')
    c = [n // 2 for n in size]
    c[up] = min(size[up] // 2 + 5, size[up] - case['pml'] - 3)
    for n in flat:
        c[n] = 0
    pol = 'xyz'[flat[0]] if flat else 'z'
    if case['source'] == 'voltage':
        b.add_voltage_source(pol, c, 50.0, 'w')
    elif case['source'] == 'magnetic':
        b.add_magnetic_dipole('xyz'[[n for n in range(3) if n not in flat][0]], c, 'w')
    else:
        b.add_hertzian_dipole(pol, c, 'w')
    along = [n for n in range(3) if n not in flat][0]
    for step in (-6, -3, 2, 4, 7):
        r = list(c)
        r[along] = min(max(r[along] + step, 0), size[along] - 1)
        b.add_rx(r)
    # one snapshot of the plane through the source, at the last iteration
    lo, hi = [0, 0, 0], list(size)
    cut = [n for n in range(3) if n not in flat][1]
    if not flat:
        lo[cut], hi[cut] = c[cut], c[cut] + 1
    b.add_snapshot(*lo, *hi, 1, 1, 1, case['its'])
    return b.finalise()


def _trace(case, seed, t):
    """Trace t of a B-scan: its own domain, soil below, dipole and receiver."""
    rng = np.random.default_rng([seed, t])
    # the domains' sides belong to the survey; the ground to the seed
    nx, ny, nz = (int(v) for v in np.random.default_rng([case['its'], t]).integers(case['lo'], case['hi'] + 1, 3))
    b = ModelBuilder(nx, ny, nz, 1e-3, 1e-3, 1e-3, case['its'], pml_cells=10)
    mats = _materials(b, rng, 64, lossy=False)
    mask = np.zeros((nx, ny, nz), dtype=bool)
    mask[:, :, :nz // 2] = True
    ids = np.ones((nx, ny, nz), dtype=np.uint32)
    ids[mask] = rng.integers(mats[0].numID, mats[0].numID + 64, int(mask.sum()), dtype=np.uint32)
    b.paint_voxels(mask, ids)
    b.add_waveform('ricker', 1, 2.5e9, 'w')
    xs = 15 + (2 * t) % (nx - 40)
    b.add_hertzian_dipole('z', (xs, ny // 2, nz // 2 + 5), 'w')
    b.add_rx((xs + 10, ny // 2, nz // 2 + 5))
    return b.finalise()


def _inversion(case, seed):
    """Start model, poles, source, receivers, wave and observed traces."""
    rng = np.random.default_rng(seed)
    shape = (case['nx'], case['ny'], case['nz'])
    er = 7.0 + 0.5 * rng.standard_normal(shape).clip(-2, 2)
    se = 1.05e-2 * (1 + 0.1 * rng.standard_normal(shape).clip(-2, 2))
    deltaer = tau = None
    if case['poles']:
        P = case['poles']
        where = rng.random(shape) < 0.4
        deltaer = rng.uniform(0.5, 5, (P,) + shape) * where
        tau = 10 ** rng.uniform(-11, -8, (P,) + shape)
    top = case['nz'] - 10 - 3
    src = (case['nx'] // 2, case['ny'] // 2, top)
    n = 16 if min(shape) > 60 else 6
    rx = [(int(x), case['ny'] // 2 + 2, top) for x in np.linspace(12, case['nx'] - 13, n)]
    dt = 2e-3 / (299792458.0 * 3 ** 0.5)
    t = np.arange(case['its']) * dt
    amp = float(rng.uniform(0.5, 2))

    def ricker(u, f=1.5e9):
        a = (np.pi * f * (u - 2 ** 0.5 / f)) ** 2
        return (1 - 2 * a) * np.exp(-a)

    waves = (amp * ricker(t)).astype(np.float32)
    dist = np.array([np.hypot(r[0] - src[0], r[1] - src[1]) * 2e-3 for r in rx])
    observed = np.stack([-300.0 * amp / (1 + 50 * q) * ricker(t - 2.6 * q / 299792458.0) for q in dist])
    return er, se, deltaer, tau, src, rx, waves, observed


def _inversion_grid(case):
    return InversionGrid((case['nx'], case['ny'], case['nz']), 2e-3, case['its'], pml=10, er_pml=7.0, K=case['K'])


def prepare(case, seed):
    if case['kind'] == 'bscan':
        return {'kind': 'bscan', 'grids': [_trace(case, seed, t) for t in range(case['traces'])]}
    if case['kind'] == 'gradient':
        er, se, deltaer, tau, src, rx, waves, observed = _inversion(case, seed)
        g = _inversion_grid(case)
        if case['poles']:
            g.set_debye(deltaer, tau)
        g.set_model(er, se)
        return {'kind': 'gradient', 'grid': g, 'src': src, 'rx': rx, 'waves': waves, 'observed': observed}
    G = _grid(case, seed)
    if case['kind'] == 'solve':
        return {'kind': 'solve', 'G': G}
    return {'kind': 'steps', 'solver': HipSolver(G), 'its': case['its']}


def run(state):
    if state['kind'] == 'bscan':
        return solve_bscan(state['grids'])[0]
    if state['kind'] == 'gradient':
        g = state['grid']
        traces = g.forward(state['src'], state['rx'], state['waves'])
        ger, gse = g.backward(traces - state['observed'])
        return [traces, ger, gse]
    if state['kind'] == 'solve':
        G = state['G']
        solve_hip(1, 1, G)
        rx = np.stack([np.stack([r.outputs[c] for r in G.rxs], axis=1) for c in ('Ex', 'Ey', 'Ez', 'Hx', 'Hy', 'Hz')])
        return [rx, G.snapshots[0].electric, G.snapshots[0].magnetic]
    s = state['solver']
    s.run(0, state['its'])
    return [s.download_rx(), s.download_snapshot(0)]


# ------------------------------------------------------------------ work
def _pml_cells(n, t):
    """Slab cells of the six faces (a face across an axis of one cell has none)."""
    return sum(2 * t * n[0] * n[1] * n[2] // n[a] for a in range(3) if n[a] > 1)


def _step_work(n, its, order, pml, poles, share, complex_):
    """One iteration reads and writes six float32 components and reads the
    three electric and three magnetic indices (2 bytes each) of every cell,
    reads and writes two Phi per slab cell, field and term, and three
    auxiliary values per pole of the dispersive cells."""
    cells = n[0] * n[1] * n[2]
    slab = _pml_cells(n, pml)
    t = 3 * poles * share * cells * (2 if complex_ else 1)
    return {'bytes': float(its * (60 * cells + 32 * order * slab + 8 * t)),
            'flops': float(its * (42 * cells + 28 * order * slab + 8 * t))}


def work(case):
    if case['kind'] == 'bscan':
        w = {'bytes': 0.0, 'flops': 0.0}
        for t in range(case['traces']):
            n = [int(v) for v in np.random.default_rng([case['its'], t]).integers(case['lo'], case['hi'] + 1, 3)]
            one = _step_work(n, case['its'], 1, 10, 0, 0, False)
            w = {k: w[k] + one[k] for k in w}
        return w
    n = (case['nx'], case['ny'], case['nz'])
    if case['kind'] == 'gradient':
        # forward, the same again for the states the adjoint needs, and the
        # adjoint: its fields, the saved E and curl, two gradients a cell
        cells, slab, P = n[0] * n[1] * n[2], _pml_cells(n, 10), case['poles']
        fwd = 60 * cells + 32 * slab + (24 + 12) * P * cells
        adj = (48 + 24 + 16 + 12) * cells + 32 * slab + ((24 + 12) * P + (12 if P else 0)) * cells
        return {'bytes': float(case['its'] * (2 * fwd + 24 * cells + adj)),
                'flops': float(case['its'] * (3 * 42 + 24 + 60 * P) * cells)}
    return _step_work(n, case['its'], case['order'], case['pml'], case['poles'], case['share'],
                      case['ground'] == 'lorentz')


# ------------------------------------------------------------------ 64 bits
# The same runs in float64 with plain torch, from the built inputs alone: the
# indices, the tables, the slabs' profiles, the sources' samples.
def _device():
    return torch.device('cuda' if torch.cuda.is_available() else 'cpu')


def _t(a):
    return torch.as_tensor(np.asarray(a), dtype=torch.float64, device=_device())


# (corrected component, source component, sign) of a slab's Phi1 and Phi2
_E_TERMS = {0: ((1, 2, -1), (2, 1, 1)), 1: ((0, 2, 1), (2, 0, -1)), 2: ((0, 1, -1), (1, 0, 1))}
_H_TERMS = {0: ((1, 2, 1), (2, 1, -1)), 1: ((0, 2, -1), (2, 0, 1)), 2: ((0, 1, 1), (1, 0, -1))}


def _slab(p, electric):
    """Cells of a slab that the field's correction touches, their neighbours
    along the normal and the profiles in the order of the cells."""
    axis = 'xyz'.index(p.direction[0])
    lo, hi = [p.xs, p.ys, p.zs], [p.xf, p.yf, p.zf]
    minus = p.direction.endswith('minus')
    off = 1 if minus and electric else 0
    t = hi[axis] - lo[axis]
    cells = [slice(a, b) for a, b in zip(lo, hi)]
    cells[axis] = slice(lo[axis] + off, lo[axis] + off + t)
    other = list(cells)
    shift = -1 if electric else 1
    other[axis] = slice(cells[axis].start + shift, cells[axis].stop + shift)
    shape = [1, 1, 1]
    shape[axis] = t
    tables = []
    for name in ('RA', 'RB', 'RE', 'RF'):
        r = _t(getattr(p, ('E' if electric else 'H') + name))
        r = r.flip(1) if minus else r
        tables.append([v.reshape(shape) for v in r])
    return axis, tuple(cells), tuple(other), tables, [b - a for a, b in zip(lo, hi)]


def _correct(mripml, R, d, src_minus, c, ph):
    """The correction of one component and its new Phi values."""
    RA, RB, RE, RF = R
    dd = src_minus / d
    if not mripml:
        if len(RA) == 1:
            return c * ((RA[0] - 1) * dd + RB[0] * ph[0]), [RE[0] * ph[0] - RF[0] * dd]
        corr = c * ((RA[0] * RA[1] - 1) * dd + RA[1] * RB[0] * ph[0] + RB[1] * ph[1])
        return corr, [RE[0] * ph[0] - RF[0] * dd, RE[1] * ph[1] - RF[1] * (RA[0] * dd + RB[0] * ph[0])]
    ira = 1 / sum(RA)
    psi = sum(b * p for b, p in zip(RB, ph))
    return (c * ((ira - 1) * dd - ira * psi),
            [RE[n] * ph[n] + ira * RF[n] * (dd - psi) if len(RA) == 2 else
             RE[n] * ph[n] + ira * RB[n] * RF[n] * (dd - ph[n]) for n in range(len(RA))])


def _ranges(nx, ny, nz):
    s = slice
    e = [(s(0, nx), s(1, ny), s(1, nz)), (s(1, nx), s(0, ny), s(1, nz)), (s(1, nx), s(1, ny), s(0, nz))]
    h = [(s(1, nx + 1), s(0, ny), s(0, nz)), (s(0, nx), s(1, ny + 1), s(0, nz)), (s(0, nx), s(0, ny), s(1, nz + 1))]
    return e, h


def _moved(r, axis, by):
    r = list(r)
    r[axis] = slice(r[axis].start + by, r[axis].stop + by)
    return tuple(r)


def _exact_solve(G):
    """Receiver buffer [6][iterations][receivers] and the first snapshot's
    six components (or None) of a grid, from zero fields."""
    nx, ny, nz = G.nx, G.ny, G.nz
    shape = (nx + 1, ny + 1, nz + 1)
    dev = _device()
    F = [torch.zeros(shape, dtype=torch.float64, device=dev) for _ in range(6)]
    ID = torch.as_tensor(G.ID.astype(np.int32), device=dev)
    cE, cH = _t(G.updatecoeffsE), _t(G.updatecoeffsH)
    er, hr = _ranges(nx, ny, nz)
    coef = []  # per component on its range: own, and the two curl factors
    for c in range(6):
        tab, r = (cE, er[c]) if c < 3 else (cH, hr[c - 3])
        m = ID[c][r].long()
        u, v = (c + 1) % 3, (c + 2) % 3
        coef.append([tab[m, q] for q in (0, 1 + u, 1 + v)])
    P = G.maxpoles
    T, dcoef = [], []
    if P:
        D = torch.as_tensor(np.asarray(G.updatecoeffsdispersive), dtype=torch.complex128, device=dev)
        D = D if G.updatecoeffsdispersive.imag.any() else D.real
        for c in range(3):
            m = ID[c][er[c]].long()
            dcoef.append([D[m, q] for q in range(3 * P)])
            T.append([torch.zeros_like(dcoef[c][0]) for _ in range(P)])
        srce = [cE[ID[c][er[c]].long(), 4] for c in range(3)]
    slabs = []
    for p in G.pmls:
        both = []
        for electric in (True, False):
            axis, cells, other, R, n = _slab(p, electric)
            tab = cE if electric else cH
            terms = (_E_TERMS if electric else _H_TERMS)[axis]
            cs = [tab[ID[(0 if electric else 3) + comp][cells].long(), 4] for comp, _, _ in terms]
            ph = [[torch.zeros(n, dtype=torch.float64, device=dev) for _ in p.CFS] for _ in terms]
            both.append((axis, cells, other, R, terms, cs, ph, p.d))
        slabs.append(both)
    del ID
    mripml = G.pmlformulation == 'MRIPML'

    def pml(both, electric):
        axis, cells, other, R, terms, cs, ph, d = both
        own, src = (F[:3], F[3:]) if electric else (F[3:], F[:3])
        for w, (comp, s, sign) in enumerate(terms):
            dd = src[s][cells] - src[s][other] if electric else src[s][other] - src[s][cells]
            corr, ph[w] = _correct(mripml, R, d, dd, cs[w], ph[w])
            own[comp][cells] += sign * corr

    rx = torch.zeros((6, G.iterations, len(G.rxs)), dtype=torch.float64, device=dev)
    at = [torch.as_tensor([getattr(r, q) for r in G.rxs], device=dev) for q in ('xcoord', 'ycoord', 'zcoord')]
    snap = None
    V = G.dx * G.dy * G.dz
    for it in range(G.iterations):
        for c in range(6):
            rx[c, it] = F[c][at[0], at[1], at[2]]
        for s in G.snapshots[:1]:
            if s.time == it + 1:
                snap = _exact_snapshot(s, F)
        for c in range(3):
            u, v = (c + 1) % 3, (c + 2) % 3
            r, (a, bu, bv) = hr[c], coef[3 + c]
            F[3 + c][r] = (a * F[3 + c][r] - bu * (F[v][_moved(r, u, 1)] - F[v][r])
                           + bv * (F[u][_moved(r, v, 1)] - F[u][r]))
        for both in slabs:
            pml(both[1], False)
        for s in G.magneticdipoles:
            i, j, k = s.xcoord, s.ycoord, s.zcoord
            c = 'xyz'.index(s.polarisation)
            F[3 + c][i, j, k] -= float(cH[int(G.ID[3 + c, i, j, k]), 4]) * float(s.waveformvalues_halfstep[it]) / V
        phis = []
        for c in range(3 if P else 0):
            e, k = F[c][er[c]], dcoef[c]
            phi = 0
            for p in range(P):
                phi = phi + (k[3 * p].real * T[c][p].real if T[c][p].is_complex() else k[3 * p] * T[c][p])
                T[c][p] = k[3 * p + 1] * T[c][p] + k[3 * p + 2] * e
            phis.append(srce[c] * phi)
        for c in range(3):
            u, v = (c + 1) % 3, (c + 2) % 3
            r, (a, bu, bv) = er[c], coef[c]
            F[c][r] = (a * F[c][r] + bu * (F[3 + v][r] - F[3 + v][_moved(r, u, -1)])
                       - bv * (F[3 + u][r] - F[3 + u][_moved(r, v, -1)]) - (phis[c] if P else 0))
        for both in slabs:
            pml(both[0], True)
        for s in G.voltagesources:
            i, j, k = s.xcoord, s.ycoord, s.zcoord
            c = 'xyz'.index(s.polarisation)
            area = V / (G.dx, G.dy, G.dz)[c]
            F[c][i, j, k] -= float(cE[int(G.ID[c, i, j, k]), 4]) * float(s.waveformvalues_wholestep[it]) / (
                s.resistance * area)
        for s in G.hertziandipoles:
            i, j, k = s.xcoord, s.ycoord, s.zcoord
            c = 'xyz'.index(s.polarisation)
            F[c][i, j, k] -= float(cE[int(G.ID[c, i, j, k]), 4]) * float(s.waveformvalues_wholestep[it]) * s.dl / V
        for c in range(3 if P else 0):
            for p in range(P):
                T[c][p] = T[c][p] - dcoef[c][3 * p + 2] * F[c][er[c]]
    return rx, snap


def _exact_snapshot(s, F):
    """Cell averages: four edges for E, two faces for H."""
    def at(a, b, c):
        return tuple(slice(o + q, o + n + q) for o, n, q in zip((s.xs, s.ys, s.zs), (s.nx, s.ny, s.nz), (a, b, c)))
    Ex, Ey, Ez, Hx, Hy, Hz = F
    return [(Ex[at(0, 0, 0)] + Ex[at(0, 1, 0)] + Ex[at(0, 0, 1)] + Ex[at(0, 1, 1)]) / 4,
            (Ey[at(0, 0, 0)] + Ey[at(1, 0, 0)] + Ey[at(0, 0, 1)] + Ey[at(1, 0, 1)]) / 4,
            (Ez[at(0, 0, 0)] + Ez[at(1, 0, 0)] + Ez[at(0, 1, 0)] + Ez[at(1, 1, 0)]) / 4,
            (Hx[at(0, 0, 0)] + Hx[at(1, 0, 0)]) / 2, (Hy[at(0, 0, 0)] + Hy[at(0, 1, 0)]) / 2,
            (Hz[at(0, 0, 0)] + Hz[at(0, 0, 1)]) / 2]


def _exact_gradient(case, seed):
    from torch.utils.checkpoint import checkpoint
    er, se, deltaer, tau, src, rx, waves, observed = _inversion(case, seed)
    g = _inversion_grid(case)
    slabs, dt, d, interior = g.slabs, g.dt, g.d, torch.as_tensor(g.interior, device=_device())
    g.close()
    e0, mu0 = 8.8541878128e-12, 1.25663706127e-6
    nx, ny, nz, P = case['nx'], case['ny'], case['nz'], case['poles']
    er, se = _t(er).requires_grad_(), _t(se).requires_grad_()
    a = e0 / dt
    Z = 0
    dk = None
    if P:
        w, q = deltaer / tau, -1.0 / tau
        zt = (w / q) * (1 - np.exp(q * dt)) / dt
        Z = _t((e0 / dt) * ((w / q) * (1 - np.exp(q * dt / 2))).sum(axis=0))
        dk = [_t(e0 * np.exp(q * dt / 2)), _t(np.exp(q * dt)), _t(zt)]
    EA, EB = a * er + 0.5 * se - Z, a * er - 0.5 * se - Z
    IEA = 1 / EA
    CA, CB = EB * IEA, IEA / d
    DB = dt / (mu0 * d)
    eR, hR = _ranges(nx, ny, nz)
    geo = [(_slab(p, True), _slab(p, False)) for p in slabs]
    shape = (nx + 1, ny + 1, nz + 1)
    dev = _device()
    zero = lambda n: torch.zeros(n, dtype=torch.float64, device=dev)  # noqa: E731
    F = [zero(shape) for _ in range(6)]
    Phi = [zero(gg[0][4]) for gg in geo for _ in range(4)]
    T = [zero(shape)[eR[c]] for c in range(3) for _ in range(P)]
    ri = [torch.as_tensor([r[q] for r in rx], device=dev) for q in range(3)]
    # cells whose coefficient enters a slab's correction: not differentiated
    IEAs = [IEA.detach()[gg[0][1]] for gg in geo]

    def slab(own, source, gg, terms, cs, ph, electric):
        axis, cells, other, R, _ = gg
        new = []
        for w, (comp, s, sign) in enumerate(terms[axis]):
            dd = source[s][cells] - source[s][other] if electric else source[s][other] - source[s][cells]
            corr, p1 = _correct(False, R, d, dd, cs, [ph[w]])
            new.append(p1[0])
            f = own[comp].clone()
            f[cells] = own[comp][cells] + sign * corr
            own[comp] = f
        return new

    def steps(n0, n1, CA, CB, IEA, *st):
        E, H = list(st[:3]), list(st[3:6])
        Phi, T = list(st[6:6 + 4 * len(geo)]), list(st[6 + 4 * len(geo):])
        out = []
        for it in range(n0, n1):
            out.append(E[2][ri[0], ri[1], ri[2]])
            nH = []
            for c in range(3):
                u, v = (c + 1) % 3, (c + 2) % 3
                r, f = hR[c], H[c].clone()
                f[r] = H[c][r] - DB * (E[v][_moved(r, u, 1)] - E[v][r]) + DB * (E[u][_moved(r, v, 1)] - E[u][r])
                nH.append(f)
            for n, gg in enumerate(geo):
                Phi[4 * n + 2:4 * n + 4] = slab(nH, E, gg[1], _H_TERMS, dt / mu0, Phi[4 * n + 2:4 * n + 4], False)
            H = nH
            nE, nT = [], []
            for c in range(3):
                u, v = (c + 1) % 3, (c + 2) % 3
                r, f = eR[c], E[c].clone()
                new = (CA[r] * E[c][r] + CB[r] * (H[v][r] - H[v][_moved(r, u, -1)])
                       - CB[r] * (H[u][r] - H[u][_moved(r, v, -1)]))
                for p in range(P):
                    t = T[c * P + p]
                    new = new - IEA[r] * dk[0][p][r] * t
                    nT.append(dk[1][p][r] * t + dk[2][p][r] * E[c][r])
                f[r] = new
                nE.append(f)
            for n, gg in enumerate(geo):
                Phi[4 * n:4 * n + 2] = slab(nE, H, gg[0], _E_TERMS, IEAs[n], Phi[4 * n:4 * n + 2], True)
            f = nE[2].clone()
            i, j, k = src
            f[i, j, k] = nE[2][i, j, k] - IEA[i, j, k] * float(waves[it]) / (d * d)
            nE[2] = f
            T = [nT[c * P + p] - dk[2][p][eR[c]] * nE[c][eR[c]] for c in range(3) for p in range(P)]
            E = nE
        return (torch.stack(out, 1), *E, *H, *Phi, *T)

    st, traces = (*F, *Phi, *T), []
    for n0 in range(0, case['its'], 16):
        got = checkpoint(steps, n0, min(n0 + 16, case['its']), CA, CB, IEA, *st, use_reentrant=False)
        traces.append(got[0])
        st = got[1:]
    traces = torch.cat(traces, 1)
    loss = 0.5 * ((traces - _t(observed)) ** 2).sum()
    ger, gse = torch.autograd.grad(loss, (er, se))
    return [traces.detach(), ger * interior, gse * interior]


def exact(case, seed):
    if case['kind'] == 'gradient':
        if case['nx'] * case['ny'] * case['nz'] * case['its'] > 2.0e9:
            return None
        return _exact_gradient(case, seed)
    if case['kind'] == 'bscan':
        return [_exact_solve(_trace(case, seed, t))[0] for t in range(case['traces'])]
    if case['nx'] * case['ny'] * case['nz'] * case['its'] > 1.2e10:
        return None
    rx, snap = _exact_solve(_grid(case, seed))
    if case['kind'] == 'solve':
        flat = [torch.stack(snap[q:q + 3]).permute(3, 2, 1, 0).reshape(-1) for q in (0, 3)]
        return [rx, flat[0], flat[1]]
    return [rx, torch.stack(snap)]
