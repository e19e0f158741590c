"""Performance cases of the FDTD stepper: what they are, how a pass over one runs, what it cannot do without, and the
same result in 64 bits.

A case is a dict of plain values. `prepare` builds the model a program holds before it steps (materials, sources,
monitors, device engine, fields of an earlier chunk of the run), `run` advances it through the public entry points
(`Simulation.run`, `Simulation3D.run`, `Batch2D.run`, `Batch3D.run`) and returns the new fields with the spectra and
probe samples taken on the way. Each pass continues the run where the last one stopped.

Geometry is laid on cell edges, so the cells of every rectangle and box are known without a raster rule; `exact` steps
the same Yee discretisation in float64 with plain torch.
"""
import math

import numpy as np
import torch

C0 = 299792458.0
EPS0 = 8.8541878128e-12
MU0 = 1.2566370614e-6
ETA0 = math.sqrt(MU0 / EPS0)
DRUDE = dict(omega_p=1.5e15, gamma=1e14, eps_inf=4.0)

PLANE = {'kind': '2d', 'pol': 'ez', 'nx': 512, 'ny': 512, 'npml': 12, 'dx': 25e-9, 'rects': 40, 'steps': 100, 'graph': 0,
         'periodic_y': False, 'flux': True, 'drude': False, 'dft': 0, 'probes': 0, 'flush': True}
SPACE = {'kind': '3d', 'nx': 128, 'ny': 128, 'nz': 128, 'npml': 8, 'dx': 25e-9, 'rects': 20, 'steps': 50, 'graph': 0,
         'flux': True, 'dft': False, 'probes': 0}


def listed():
    return [
        # the thin-film transmission run of the examples, start to end (80 fs), one spectrum read after it
        {**PLANE, 'name': 'film_ez', 'nx': 270, 'ny': 120, 'npml': 15, 'rects': 1, 'steps': 1370, 'periodic_y': True},
        # the same film in the other polarisation, stepped by replayed graphs
        {**PLANE, 'name': 'film_hz', 'pol': 'hz', 'nx': 270, 'ny': 120, 'npml': 15, 'rects': 1, 'steps': 1370,
         'periodic_y': True, 'graph': 50},
        # a coupled run: a few steps between callbacks, nothing waited for; launches and host work are all there is
        {**PLANE, 'name': 'coupled_chunk', 'nx': 190, 'ny': 157, 'rects': 6, 'steps': 8, 'flux': False, 'flush': False},
        # one model of a parameter sweep, an odd grid of ordinary size with the default options
        {**PLANE, 'name': 'sweep_ez', 'nx': 1031, 'ny': 773, 'rects': 60, 'steps': 300},
        # a larger ordinary H_z model replayed from graphs
        {**PLANE, 'name': 'guide_hz', 'pol': 'hz', 'nx': 1500, 'ny': 1102, 'rects': 80, 'steps': 200, 'graph': 50},
        # metal, near-field spectra over a box and probes: every per-step extra of a scattering study
        {**PLANE, 'name': 'metal_ez', 'nx': 2048, 'ny': 2050, 'rects': 60, 'steps': 100, 'drude': True, 'dft': 4,
         'probes': 16},
        # the large E_z grid of the benchmark, replayed from graphs
        {**PLANE, 'name': 'large_ez', 'nx': 8192, 'ny': 8192, 'npml': 20, 'dx': 20e-9, 'rects': 400, 'steps': 40,
         'graph': 20, 'flux': False},
        # a large H_z grid of odd sides with the default options
        {**PLANE, 'name': 'large_hz', 'pol': 'hz', 'nx': 4099, 'ny': 5003, 'npml': 20, 'dx': 20e-9, 'rects': 200,
         'steps': 30},
        # a small 3D antenna model: dipole, flux plane, near-field plane, probes
        {**SPACE, 'name': 'antenna_3d', 'nx': 97, 'ny': 88, 'nz': 75, 'steps': 100, 'dft': True, 'probes': 4},
        # the large 3D grid of the benchmark, replayed from graphs
        {**SPACE, 'name': 'large_3d', 'nx': 512, 'ny': 512, 'nz': 512, 'npml': 12, 'rects': 200, 'steps': 8, 'graph': 4},
        # uneven 2D models of both polarisations stepped together, as a sweep or the server's chunks do
        {'name': 'batch_2d', 'kind': 'batch2d', 'members': 28, 'lo': 128, 'hi': 1024, 'npml': 12, 'steps': 200},
        # uneven 3D models stepped together
        {'name': 'batch_3d', 'kind': 'batch3d', 'members': 6, 'lo': 64, 'hi': 140, 'npml': 8, 'steps': 60},
    ]


def draw(rng):
    """One more case of the ranges above: grids of 100 to 8192 cells a side in 2D, 40 to 512 in 3D, 1 to 1500 steps."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(['2d', '2d', '2d', '2d', '3d', '3d', 'batch2d', 'batch3d'])
    if kind == '2d':
        nx, ny = log_int(100, 8192), log_int(100, 8192)
        most = max(1, min(1500, 2_600_000_000 // (nx * ny)))
        drude = rng.random() < 0.2
        pol = 'ez' if drude else rng.choice(['ez', 'hz'])
        return {**PLANE, 'pol': pol, 'nx': nx, 'ny': ny, 'npml': rng.choice([10, 12, 15, 20]),
                'rects': log_int(4, 200), 'steps': log_int(1, most), 'graph': rng.choice([0, 0, 10, 50]),
                'periodic_y': rng.random() < 0.25, 'flux': rng.random() < 0.7, 'drude': drude,
                'dft': rng.choice([0, 0, 0, 3]), 'probes': rng.choice([0, 0, 5])}
    if kind == '3d':
        nx, ny, nz = (log_int(40, 512) for _ in range(3))
        most = max(1, min(300, 1_000_000_000 // (nx * ny * nz)))
        return {**SPACE, 'nx': nx, 'ny': ny, 'nz': nz, 'npml': rng.choice([8, 10, 12]), 'rects': log_int(4, 60),
                'steps': log_int(1, most), 'graph': rng.choice([0, 0, 10]), 'flux': rng.random() < 0.7,
                'dft': rng.random() < 0.3, 'probes': rng.choice([0, 3])}
    if kind == 'batch2d':
        return {'kind': kind, 'members': rng.randint(2, 28), 'lo': 100, 'hi': log_int(200, 1024), 'npml': 12,
                'steps': log_int(10, 300)}
    return {'kind': kind, 'members': rng.randint(2, 8), 'lo': 40, 'hi': log_int(60, 140), 'npml': 8,
            'steps': log_int(10, 100)}


# ---- the scene: everything that follows from a case and a seed, in whole cells --------------------------------------
def rng_of(case, seed):
    return np.random.default_rng([int(seed), case['nx'], case['ny'], case.get('nz', 0), case['steps']])


def f32(value):
    return float(np.float32(value))


def waves_along(rng, n, lo, hi, count):
    """(n, count) float32 waves along one axis, faded to 0 at both ends of the window [lo, hi)."""
    s = np.arange(n) - lo
    size = hi - lo
    fade = np.where((s >= 0) & (s < size), np.sin(np.pi * (s + 0.5) / size) ** 2, 0.0)
    wavelength = rng.uniform(12.0, 60.0, count)
    phase = rng.uniform(0.0, 2 * np.pi, count)
    return (fade[:, None] * np.sin(2 * np.pi * s[:, None] / wavelength + phase)).astype(np.float32)


class Scene:
    """A model in whole cells: window, rectangles or boxes, source, monitors and the fields it starts from."""

    def __init__(self, case, seed):
        self.case = case
        rng = rng_of(case, seed)
        self.dims = 3 if case['kind'] == '3d' else 2
        self.shape = tuple(case[k] for k in ('nx', 'ny', 'nz')[:self.dims])
        self.npml, self.dx, self.steps = case['npml'], case['dx'], case['steps']
        self.periodic = (False, bool(case.get('periodic_y')), False)[:self.dims]
        self.pad = tuple(0 if p else self.npml for p in self.periodic)
        self.window = tuple(n - 2 * p for n, p in zip(self.shape, self.pad))
        self.boxes = []   # (lo per axis, hi per axis, eps_r) in window cells, later ones over earlier ones
        if case['rects'] == 1:   # the film: a slab across the window
            third = self.window[0] // 3
            self.boxes.append(((third, 0), (third + self.window[0] // 12, self.window[1]), 2.25))
        else:
            for _ in range(case['rects']):
                size = [max(2, int(w * rng.uniform(0.03, 0.3))) for w in self.window]
                lo = [int(rng.integers(1, max(2, w - s - 1))) for w, s in zip(self.window, size)]
                hi = [min(w - 1, a + s) for w, a, s in zip(self.window, lo, size)]
                self.boxes.append((tuple(lo), tuple(hi), f32(rng.uniform(1.0, 12.0))))
        self.wavelength = rng.uniform(20.0, 40.0) * self.dx
        self.wavelengths = [0.9 * self.wavelength, self.wavelength, 1.1 * self.wavelength]
        w = self.window
        self.source = w[0] // 4 if self.dims == 2 else tuple(n // 2 for n in w)
        self.flux_at = 3 * w[0] // 4
        self.dft_layer = w[2] // 3 if self.dims == 3 else 0
        self.metal = ((w[0] // 2, w[1] // 4), (w[0] // 2 + max(1, w[0] // 6), 3 * w[1] // 4))
        self.probes = [tuple(int(rng.integers(0, n)) for n in w) for _ in range(case['probes'])]
        self.names = (('ex', 'ey', 'ez', 'hx', 'hy', 'hz') if self.dims == 3 else
                      ('ez', 'hx', 'hy') if case['pol'] == 'ez' else ('hz', 'ex', 'ey'))
        self.modes = {}
        for name in self.names:
            along = [waves_along(rng, n, p, n - p, 4) for n, p in zip(self.shape, self.pad)]
            along[0] *= np.float32(1.0 if name[0] == 'e' else 1.0 / ETA0)
            self.modes[name] = [torch.from_numpy(a) for a in along]
        # the float32 cell width and time step of the model are part of its definition
        self.width = f32(self.dx)
        d = self.dx if self.dims == 2 else self.width
        self.dt = f32(0.99 / (C0 * math.sqrt(sum(1.0 / d ** 2 for _ in self.shape))))

    def field(self, name):
        """float32 field `name` at the start of the first pass, on the host."""
        a = self.modes[name]
        if self.dims == 2:
            return a[0] @ a[1].T
        return (a[0] @ (a[1][:, None, :] * a[2][None, :, :]).reshape(-1, a[0].shape[1]).T).reshape(self.shape)

    def sample_interval(self):
        """Steps between spectrum samples: the Nyquist bound of the source's and the monitors' highest frequencies."""
        if not (self.case['flux'] or self.case['dft']):
            return 1
        rate = C0 / self.wavelength * (1.0 + 3.72 * 0.5) + C0 / min(self.wavelengths)
        return max(1, int(math.floor(1.0 / (rate * self.dt))))


# ---- models on the device ---------------------------------------------------------------------------------------
def build_2d(case, scene):
    from opensol_amd import DrudePole, Simulation
    dx, w = scene.dx, scene.window
    sim = Simulation(w[0] * dx, w[1] * dx, dx, npml=scene.npml, boundaries='periodic_y' if scene.periodic[1] else None,
                     polarization=case['pol'], graph_steps=case['graph'])
    for lo, hi, eps in scene.boxes:
        sim.add_dielectric_rectangle(lo[0] * dx, lo[1] * dx, hi[0] * dx, hi[1] * dx, eps_r=eps)
    if case['drude']:
        lo, hi = scene.metal
        sim.add_drude_rectangle(lo[0] * dx, lo[1] * dx, hi[0] * dx, hi[1] * dx, DrudePole(**DRUDE))
    sim.add_line_source(axis='y', position=(scene.source + 0.5) * dx, wavelength=scene.wavelength, bandwidth=0.5)
    if case['flux']:
        sim.add_flux_monitor(axis='y', position=(scene.flux_at + 0.5) * dx, span=(0.0, w[1] * dx),
                             wavelengths=scene.wavelengths)
    if case['dft']:
        sim.add_dft_monitor(0.5 * dx, 0.5 * dx, (w[0] - 0.5) * dx, (w[1] - 0.5) * dx, wavelengths=scene.wavelengths,
                            downsample=case['dft'])
    for i, j in scene.probes:
        sim.add_field_probe((i + 0.5) * dx, (j + 0.5) * dx)
    return sim


def build_3d(case, scene):
    from opensol_amd import Simulation3D
    dx, w = scene.dx, scene.window
    sim = Simulation3D(*(n * dx for n in w), dx, npml=scene.npml, graph_steps=case['graph'])
    for lo, hi, eps in scene.boxes:
        sim.add_dielectric_box(tuple(v * dx for v in lo), tuple(v * dx for v in hi), eps_r=eps)
    x, y, z = ((v + 0.5) * dx for v in scene.source)
    sim.add_dipole(x, y, z + 0.5 * dx, orientation='z', dipole_moment=3e-18, wavelength=scene.wavelength,
                   bandwidth=0.5)
    if case['flux']:
        sim.add_flux_plane('x', scene.flux_at * dx, wavelengths=scene.wavelengths)
    if case['dft']:
        sim.add_dft_plane((scene.dft_layer + 0.5) * dx, wavelengths=scene.wavelengths)
    for i, j, k in scene.probes:
        sim.add_field_probe((i + 0.5) * dx, (j + 0.5) * dx, (k + 0.5) * dx)
    return sim


def build(case, seed):
    """The simulation of a single-model case: device engine built, tables for the coming steps laid out, fields set."""
    scene = Scene(case, seed)
    sim = (build_3d if scene.dims == 3 else build_2d)(case, scene)
    sim.finalize()
    assert tuple(sim.model.shape) == scene.shape, (sim.model.shape, scene.shape)
    # a run's tables are laid out once for its whole length: many chunks of `steps` steps
    sim.engine.prepare(max(4 * case['steps'], min(400 * case['steps'], 30_000)))
    for name in scene.names:
        sim.engine.set_field(name, scene.field(name))
    return sim


def member_cases(case):
    """The single-model cases of a batch, each with its own sides and step count."""
    rng = np.random.default_rng([case['members'], case['hi'], case['steps']])
    dims = 3 if case['kind'] == 'batch3d' else 2
    out = []
    for k in range(case['members']):
        sides = [int(round(math.exp(rng.uniform(math.log(case['lo']), math.log(case['hi']))))) for _ in range(dims)]
        steps = int(rng.integers((case['steps'] + 1) // 2, case['steps'] + 1)) if k else case['steps']
        base = {**(SPACE if dims == 3 else PLANE), **dict(zip(('nx', 'ny', 'nz'), sides)), 'npml': case['npml'],
                'steps': steps}
        out.append({**base, 'rects': 12} if dims == 3 else {**base, 'pol': 'ez' if k % 2 == 0 else 'hz'})
    return out


def prepare(case, seed):
    if not case['kind'].startswith('batch'):
        return {'case': case, 'sim': build(case, seed)}
    from opensol_amd.batch import Batch2D, Batch3D
    members = member_cases(case)
    sims = [build(m, int(seed) * 1000 + k) for k, m in enumerate(members)]
    batch = (Batch3D if case['kind'] == 'batch3d' else Batch2D)(sims)
    return {'case': case, 'sims': sims, 'batch': batch, 'steps': [m['steps'] for m in members]}


def spectrum(acc, axis):
    """(sum re, sum im) minus their compensations: the spectra, without leaving the device."""
    s = acc.narrow(axis, 0, 2)
    return s - acc.narrow(axis, 2, 2)


def fields_of(sim):
    """The current fields on the device, padding columns left out."""
    engine = sim.engine
    now = engine.fields[engine.n_step & 1]
    return now[..., :sim.model.ny] if now.dim() == 3 else now


def outputs(sim):
    engine = sim.engine
    out = {'fields': fields_of(sim)}
    for k, acc in enumerate(engine.accumulators):
        if isinstance(acc, list):
            for q, pair in enumerate(acc):
                out[f'flux{k}_{q}'] = spectrum(pair, 2)
        else:
            out[f'flux{k}'] = spectrum(acc, 2)
    for k, acc in enumerate(engine.dft_accumulators):
        out[f'dft{k}'] = spectrum(acc, acc.dim() - 1)
    return out


def run(state):
    case = state['case']
    if 'batch' in state:
        state['batch'].run(state['steps'])
        state['batch'].synchronize()
        return [{'fields': fields_of(s), 'flux': [spectrum(a, 2) for acc in s.engine.accumulators
                                                  for a in (acc if isinstance(acc, list) else [acc])][0]}
                for s in state['sims']]
    sim = state['sim']
    sim.run(n_steps=case['steps'], print_every=0, flush=case.get('flush', True))
    if case['rects'] == 1:   # the film run ends with its transmitted power
        return {'fields': fields_of(sim), 'flux': sim.monitors[0].flux()}
    out = outputs(sim)
    if case['probes']:
        out['probes'] = [p.get_data()[1][-case['steps']:] for p in sim.model.probes]
    return out


def work(case):
    """Fields and ids read once and the new fields written once; the additions and multiplications of the updates."""
    if case['kind'].startswith('batch'):
        parts = [work(m) for m in member_cases(case)]
        return {k: sum(p[k] for p in parts) for k in ('bytes', 'flops')}
    if case['kind'] == '2d':
        cells = case['nx'] * case['ny']
        return {'bytes': 26 * cells, 'flops': 18 * cells * case['steps']}
    cells = case['nx'] * case['ny'] * case['nz']
    return {'bytes': 50 * cells, 'flops': 48 * cells * case['steps']}


# ---- the same runs in 64 bits -----------------------------------------------------------------------------------
class Axis:
    """Stretched inverse spacings and CPML recursion factors of one axis, as float64 vectors over its rows: order 3,
    kappa up to 15, no alpha; the layers' psi rows are 1..npml (centres) and 0..npml-1 (hi faces) on the low side and
    n-npml-1..n-2 on the high side."""

    def __init__(self, scene, axis, device):
        n, npml, dx, dt = scene.shape[axis], scene.npml, scene.width, scene.dt
        self.periodic = scene.periodic[axis]
        kappa, b, g = (np.ones((2, n)), np.zeros((2, n)), np.zeros((2, n)))
        if not self.periodic:
            sigma_max = 4.0 / (150.0 * math.pi * dx)
            q = np.arange(npml, dtype=np.float64)
            sides = (((npml - 1 - q) / npml, slice(1, npml + 1), (npml - q - 0.5) / npml, slice(0, npml)),
                     (q / npml, slice(n - npml - 1, n - 1), (q + 0.5) / npml, slice(n - npml - 1, n - 1)))
            for depth_e, rows_e, depth_h, rows_h in sides:
                for kind, depth, rows in ((0, depth_e, rows_e), (1, depth_h, rows_h)):
                    sigma, k = sigma_max * depth ** 3, 1.0 + 14.0 * depth ** 3
                    factor = np.exp(-sigma / k * dt / EPS0)
                    kappa[kind, rows], b[kind, rows] = k, factor
                    g[kind, rows] = np.where(sigma > 0, (factor - 1.0) / k / dx, 0.0)
        shape = [1] * scene.dims
        shape[axis] = n

        def vector(v):
            return torch.from_numpy(np.ascontiguousarray(v)).to(device).reshape(shape)

        self.inv = [vector(1.0 / (dx * kappa[kind])) for kind in (0, 1)]
        self.b, self.g = [vector(v) for v in b], [vector(v) for v in g]
        self.axis, self.layers = axis, not self.periodic

    def up(self, f):
        """f of the next row minus f; 0 on the last row of a bounded axis."""
        if self.periodic:
            return torch.roll(f, -1, self.axis) - f
        out = torch.zeros_like(f)
        n = f.shape[self.axis]
        out.narrow(self.axis, 0, n - 1).copy_(torch.diff(f, dim=self.axis))
        return out

    def down(self, f):
        """f minus f of the row before; a bounded axis reads 0 below row 0."""
        if self.periodic:
            return f - torch.roll(f, 1, self.axis)
        out = f.clone()
        n = f.shape[self.axis]
        out.narrow(self.axis, 1, n - 1).sub_(f.narrow(self.axis, 0, n - 1))
        return out

    def derivative(self, f, kind, psi):
        """The stretched derivative of f with its psi (updated in place); kind 0 at centres, 1 on hi faces."""
        d = self.up(f) if kind else self.down(f)
        if self.layers:
            psi.mul_(self.b[kind]).add_(d * self.g[kind])
            return d * self.inv[kind] + psi
        return d * self.inv[kind]

    def face_mean(self, f):
        """Mean of f over each cell and its next one; the last face of a bounded axis takes its own cell."""
        other = torch.roll(f, -1, self.axis)
        if not self.periodic:
            n = f.shape[self.axis]
            other.narrow(self.axis, n - 1, 1).copy_(f.narrow(self.axis, n - 1, 1))
        return 0.5 * (f + other)


class Recorder:
    """Running DFT of the sampled values: sum over samples of value exp(-j omega t) m dt."""

    def __init__(self, scene, device):
        self.m, self.dt = scene.sample_interval(), scene.dt
        self.omega = 2.0 * math.pi * C0 / torch.tensor(scene.wavelengths, dtype=torch.float64, device=device)
        self.sums = {}

    def add(self, n, time, name, value):
        if (n + 1) % self.m:
            return
        phase = -self.omega * time
        factor = torch.stack([torch.cos(phase), torch.sin(phase)], dim=-1) * (self.m * self.dt)
        shape = [1] * value.dim()
        term = factor.reshape(*factor.shape, *shape) * value
        self.sums[name] = self.sums[name] + term if name in self.sums else term


def pulse(scene, t):
    """Gaussian pulse of relative bandwidth 0.5 around the scene's wavelength."""
    f0 = C0 / scene.wavelength
    tau = 1.0 / (0.5 * f0 * math.pi)
    s = t - 4.5 * tau
    return math.exp(-(s / tau) ** 2) * math.sin(2.0 * math.pi * f0 * s)


def permittivity(scene, device):
    eps = torch.ones(scene.shape, dtype=torch.float64, device=device)
    for lo, hi, value in scene.boxes:
        eps[tuple(slice(p + a, p + b) for p, a, b in zip(scene.pad, lo, hi))] = value
    return eps


def exact_2d(case, scene, device):
    hz = case['pol'] == 'hz'
    x, y = Axis(scene, 0, device), Axis(scene, 1, device)
    dt, pad = scene.dt, scene.pad
    eps = permittivity(scene, device)
    f = {name: scene.field(name).to(device=device, dtype=torch.float64) for name in scene.names}
    psi = {k: torch.zeros(scene.shape, dtype=torch.float64, device=device) for k in ('xe', 'xh', 'ye', 'yh')}
    db = dt / MU0
    metal = None
    if case['drude']:
        metal = tuple(slice(p + a, p + b) for p, a, b in zip(pad, *scene.metal))
        eps[metal] = DRUDE['eps_inf']
        denominator = 1.0 + DRUDE['gamma'] * dt / 2.0
        damping, drive = -DRUDE['gamma'] * dt / denominator, EPS0 * DRUDE['omega_p'] ** 2 * dt / denominator
        current = torch.zeros_like(eps[metal])
    line = pad[0] + scene.source
    cb_x = dt / (EPS0 * (x.face_mean(eps) if hz else eps))   # of E_y on the hi-x faces, of E_z at the centres
    cb_y = dt / (EPS0 * y.face_mean(eps)) if hz else None
    line_eps = x.face_mean(eps)[line] if hz else eps[line]
    spacing = scene.width if hz else scene.dx
    half = spacing * math.sin(math.pi * C0 / scene.wavelength * dt) / (C0 * dt)
    profile = cb_x[line] * torch.sqrt(line_eps * (1.0 - line_eps * half ** 2)) * 2.0 / (ETA0 * spacing)
    record = Recorder(scene, device)
    at, span = pad[0] + scene.flux_at, slice(pad[1], scene.shape[1] - pad[1])
    stride = case['dft']
    probes = [[] for _ in scene.probes]
    t = 0.0
    for n in range(scene.steps):
        value = pulse(scene, t + 0.5 * dt)
        if hz:
            f['hz'] += db * (y.derivative(f['ex'], 0, psi['ye']) - x.derivative(f['ey'], 0, psi['xe']))
            f['ex'] += cb_y * y.derivative(f['hz'], 1, psi['yh'])
            f['ey'] -= cb_x * x.derivative(f['hz'], 1, psi['xh'])
            f['ey'][line] += value * profile
            e, h = f['ey'], f['hz']
        else:
            f['hx'] -= db * y.derivative(f['ez'], 1, psi['yh'])
            f['hy'] += db * x.derivative(f['ez'], 1, psi['xh'])
            if metal is not None:
                current += damping * current + drive * f['ez'][metal]
            f['ez'] += cb_x * (x.derivative(f['hy'], 0, psi['xe']) - y.derivative(f['hx'], 0, psi['ye']))
            if metal is not None:
                f['ez'][metal] -= cb_x[metal] * current
            f['ez'][line] += value * profile
            e, h = f['ez'], f['hy']
        t += dt
        if case['flux']:
            record.add(n, t, 'flux', torch.stack([e[at, span], h[at, span]]))
        if stride:
            wx, wy = (slice(p + min(stride, w) // 2, p + w, stride) for p, w in zip(pad, scene.window))
            boxes = [f[scene.names[0]][wx, wy]]
            if hz:   # in-plane E at the cell centres: the mean with the face below
                boxes += [(f['ex'] - 0.5 * y.down(f['ex']))[wx, wy], (f['ey'] - 0.5 * x.down(f['ey']))[wx, wy]]
            record.add(n, t, 'dft', torch.stack(boxes))
        for k, (i, j) in enumerate(scene.probes):
            probes[k].append(f[scene.names[0]][pad[0] + i, pad[1] + j].clone())
    out = {'fields': torch.stack([f[name] for name in scene.names])}
    spectra = {k: v.movedim((2,), (0,)) for k, v in record.sums.items()}   # (component, frequency, re/im, cells)
    if case['flux']:
        out['flux0'] = spectra.get('flux', torch.zeros(2, 3, 2, scene.window[1], dtype=torch.float64))
        if case['rects'] == 1:
            out['flux'] = power_2d(case, scene, out.pop('flux0'))
    if stride and 'dft' in spectra:
        out['dft0'] = spectra['dft'].movedim(2, -1)
    if scene.probes:
        out['probes'] = [torch.stack(p) for p in probes]
    return out


def power_2d(case, scene, spectra):
    """Transmitted power at each wavelength from the (E, H) spectra of the flux line."""
    f = (C0 / torch.tensor(scene.wavelengths, dtype=torch.float64)).to(spectra.device)
    z = torch.complex(spectra[:, :, 0], spectra[:, :, 1])
    turn = torch.exp(1j * math.pi * f * scene.dt)[:, None]
    sign = 1.0 if case['pol'] == 'hz' else -1.0
    real = (z[0] * torch.conj(z[1] * turn)).real.sum(dim=1) * scene.dx
    return (sign * torch.cos(math.pi * f * scene.dt) * real).cpu().numpy()


def exact_3d(case, scene, device):
    axes = [Axis(scene, a, device) for a in range(3)]
    x, y, z = axes
    dt, pad = scene.dt, scene.pad
    eps = permittivity(scene, device)
    cb = [dt / (EPS0 * a.face_mean(eps)) for a in axes]
    db = dt / MU0
    f = {name: scene.field(name).to(device=device, dtype=torch.float64) for name in scene.names}
    psi = {}

    def d(axis, name, kind):
        key = (axis.axis, name)
        if key not in psi:
            psi[key] = torch.zeros(scene.shape, dtype=torch.float64, device=device)
        return axis.derivative(f[name], kind, psi[key])

    cell = tuple(p + s for p, s in zip(pad, scene.source))   # the dipole on the hi-z face of this cell
    weight = float(cb[2][cell]) * 3e-18 / scene.width ** 3
    record = Recorder(scene, device)
    edge = pad[0] + scene.flux_at
    wy, wz = (slice(pad[a], scene.shape[a] - pad[a]) for a in (1, 2))
    faces = [slice(pad[a], scene.shape[a] - pad[a]) for a in (1, 2)]
    layer = pad[2] + scene.dft_layer
    probes = [[] for _ in scene.probes]
    t = 0.0
    for n in range(scene.steps):
        f['hx'] -= db * (d(y, 'ez', 1) - d(z, 'ey', 1))
        f['hy'] -= db * (d(z, 'ex', 1) - d(x, 'ez', 1))
        f['hz'] -= db * (d(x, 'ey', 1) - d(y, 'ex', 1))
        f['ex'] += cb[0] * (d(y, 'hz', 0) - d(z, 'hy', 0))
        f['ey'] += cb[1] * (d(z, 'hx', 0) - d(x, 'hz', 0))
        f['ez'] += cb[2] * (d(x, 'hy', 0) - d(y, 'hx', 0))
        f['ez'][cell] += weight * pulse(scene, t + 0.5 * dt)
        t += dt
        if case['flux']:   # samples on the hi faces of the window edges first..last along the E component's own axis
            ys = slice(max(faces[0].start, 1) - 1, faces[0].stop)
            zs = slice(max(faces[1].start, 1) - 1, faces[1].stop)
            for q, (e, h, sy, sz) in enumerate((('ey', 'hz', ys, wz), ('ez', 'hy', wy, zs))):
                mean = 0.5 * (f[e][edge - 1, sy, sz] + f[e][edge, sy, sz])
                record.add(n, t, f'flux0_{q}', torch.stack([mean, f[h][edge - 1, sy, sz]]))
        if case['dft']:
            wx = slice(pad[0], scene.shape[0] - pad[0])
            centred = [(f[e] - 0.5 * axes[a].down(f[e]))[wx, wy, layer:layer + 1]
                       for a, e in enumerate(('ex', 'ey', 'ez'))]
            record.add(n, t, 'dft0', torch.stack(centred))
        for k, (i, j, m) in enumerate(scene.probes):
            probes[k].append(f['ez'][pad[0] + i, pad[1] + j, pad[2] + m].clone())
    out = {'fields': torch.stack([f[name] for name in scene.names])}
    for name, value in record.sums.items():
        value = value.movedim(2, 0)
        out[name] = value.movedim(2, -1) if name == 'dft0' else value
    if scene.probes:
        out['probes'] = [torch.stack(p) for p in probes]
    return out


def exact(case, seed):
    device = torch.device('cuda' if torch.cuda.is_available() else 'cpu')
    if case['kind'].startswith('batch'):
        members = member_cases(case)
        found = [exact_one(m, int(seed) * 1000 + k, device) for k, m in enumerate(members)]
        return [{'fields': v['fields'], 'flux': v.get('flux0', v.get('flux0_0'))} for v in found]
    return exact_one(case, seed, device)


def exact_one(case, seed, device):
    scene = Scene(case, seed)
    return (exact_3d if scene.dims == 3 else exact_2d)(case, scene, device)
