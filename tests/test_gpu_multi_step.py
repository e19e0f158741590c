"""Several 2D steps in one launch against the same steps one launch each (step_timed): every field, psi array and
accumulator equal bit for bit, at sizes around the window edges, across polarisations, boundaries, materials, sources,
monitors and step counts, from random fields and psi."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DX, NPML = 25e-9, 8


def build(pol, nx, ny, boundaries, media, graph_steps=0, extras=None):
    from opensol_amd import Simulation
    px, py = boundaries in ('periodic_x', 'periodic'), boundaries in ('periodic_y', 'periodic')
    wx, wy = nx - (0 if px else 2 * NPML), ny - (0 if py else 2 * NPML)
    sim = Simulation(wx * DX, wy * DX, DX, npml=NPML, boundaries=boundaries, polarization=pol, graph_steps=graph_steps)
    assert sim.model.shape == (nx, ny)
    rng = np.random.default_rng([nx, ny])
    for _ in range(6):
        x0, y0 = rng.uniform(0, 0.7 * wx * DX), rng.uniform(0, 0.7 * wy * DX)
        sim.add_dielectric_rectangle(x0, y0, x0 + 0.3 * wx * DX, y0 + 0.3 * wy * DX, eps_r=rng.uniform(1, 12),
                                     sigma_e=2e3 if media == 'lossy' else 0.0)
    if media == 'pec':
        sim.add_pec_rectangle(0.3 * wx * DX, 0.2 * wy * DX, 0.5 * wx * DX, 0.6 * wy * DX)
    sim.add_line_source(axis='y', position=0.4 * wx * DX, wavelength=600e-9, bandwidth=0.8, waveform='ricker')
    sim.add_line_source(axis='x', position=0.6 * wy * DX, wavelength=700e-9, bandwidth=0.8, waveform='ricker',
                        span=(0.1 * wx * DX, 0.8 * wx * DX))
    if pol == 'ez':
        sim.add_point_source(0.5 * wx * DX, 0.5 * wy * DX, wavelength=600e-9, waveform='ricker')
    else:
        sim.add_magnetic_line_current(0.5 * wx * DX, 0.5 * wy * DX, wavelength=600e-9, waveform='ricker')
        sim.add_electric_dipole(0.7 * wx * DX, 0.3 * wy * DX, wavelength=600e-9, orientation=30.0, waveform='ricker')
    sim.add_flux_monitor(axis='y', position=0.7 * wx * DX, span=(0.0, wy * DX), wavelengths=[500e-9, 700e-9])
    sim.add_flux_monitor(axis='x', position=0.2 * wy * DX, span=(0.2 * wx * DX, wx * DX), wavelengths=[600e-9])
    if extras:
        extras(sim, wx, wy)
    sim.finalize()
    torch = sim.engine.torch
    generator = torch.Generator().manual_seed(nx * 1000 + ny)

    def fill(t):   # the current set only, as a restored run has it; padding columns stay 0
        t.copy_(torch.randn(t.shape, generator=generator))
    fill(sim.engine.fields[0, :, :, :ny])
    for axis in sim.engine.cpml.values():
        if axis is not None:
            fill(axis['psi_e'][0][..., :ny] if axis is sim.engine.cpml['x'] else axis['psi_e'][0])
            fill(axis['psi_h'][0][..., :ny] if axis is sim.engine.cpml['x'] else axis['psi_h'][0])
    # psi of a hi-face row past the grid's last one is never updated and holds 0 in a run
    return sim


def arrays(sim, n):
    e = sim.engine
    out = {'fields': e.fields[n & 1]}
    for name, axis in e.cpml.items():
        if axis is not None:
            out[f'psi_e {name}'], out[f'psi_h {name}'] = axis['psi_e'][n & 1], axis['psi_h'][n & 1]
    out.update({f'acc {k}': a for k, a in enumerate(e.accumulators)})
    out['clock'] = e.clock
    return out


# sizes below, at and past one window (64 x 16, 64 x 32, 64 x 64 cells less their halos), odd columns, a few windows,
# and grids with an interior of 128 x 64 windows
SIZES = [(20, 19), (34, 64), (61, 37), (50, 108), (129, 130), (300, 257), (97, 700), (611, 523)]


@pytest.mark.parametrize('pol', ['ez', 'hz'])
@pytest.mark.parametrize('nx,ny', SIZES)
@pytest.mark.parametrize('boundaries,media', [('pml', 'plain'), ('periodic_y', 'lossy'), ('periodic_x', 'pec'),
                                              ('periodic', 'plain'), ('pml', 'lossy')])
def test_multi_step_matches_single_steps(gpu, pol, nx, ny, boundaries, media):
    multi, single = (build(pol, nx, ny, boundaries, media) for _ in range(2))
    total = 0
    for steps in (1, 2, 7, 20, 33):
        multi.engine.step(steps)
        single.engine.step_timed(steps)
        total += steps
        a, b = arrays(multi, total), arrays(single, total)
        for name in a:
            same = (a[name] == b[name]).all()
            assert bool(same), (name, total, int((a[name] != b[name]).sum()))


@pytest.mark.parametrize('pol', ['ez', 'hz'])
def test_multi_step_graph_replays(gpu, pol):
    """Graphs of an odd and an even number of steps, replayed several times with eager steps between."""
    for graph_steps in (5, 12):
        graphed, single = build(pol, 140, 171, 'pml', 'plain', graph_steps), build(pol, 140, 171, 'pml', 'plain')
        total = 0
        for steps in (2 * graph_steps, 3, graph_steps + 1, 3 * graph_steps):
            graphed.engine.step(steps)
            single.engine.step_timed(steps)
            total += steps
            a, b = arrays(graphed, total), arrays(single, total)
            for name in a:
                assert bool((a[name] == b[name]).all()), (name, graph_steps, total)


# (polarisation, nx, ny, boundaries, media): grids with and without a lean interior, of both polarisations
MEMBERS = [('ez', 61, 37, 'pml', 'plain'), ('hz', 129, 130, 'pml', 'lossy'), ('ez', 611, 523, 'periodic_y', 'lossy'),
           ('hz', 34, 64, 'periodic', 'plain'), ('ez', 300, 257, 'pml', 'pec'), ('hz', 97, 300, 'periodic_x', 'pec'),
           ('ez', 20, 19, 'periodic', 'plain')]


@pytest.mark.parametrize('graph_steps', [0, 9])
@pytest.mark.parametrize('large', [False, True])
def test_multi_step_batch_members(gpu, graph_steps, large):
    """Members that stop within, at the end of and between launches, after odd and even counts, over several calls."""
    from opensol_amd.batch import Batch2D
    chosen = [m for m in MEMBERS if large or m[1] * m[2] < 100_000] * (4 if large else 1)
    members, singles = ([build(*m) for m in chosen] for _ in range(2))
    batch = Batch2D(members, graph_steps=graph_steps)
    totals = [0] * len(chosen)
    for call in ([29, 14, 1, 22, 28, 0, 15], [3, 2, 1, 0, 3, 2, 1], [12, 11, 10, 9, 4, 12, 0], [40] * 7):
        counts = [call[k % 7] for k in range(len(chosen))]
        batch.run(counts)
        for k, (a, b, n) in enumerate(zip(members, singles, counts)):
            if n:
                b.engine.step_timed(n)
            totals[k] += n
            got, expected = arrays(a, totals[k]), arrays(b, totals[k])
            for name in got:
                assert bool((got[name] == expected[name]).all()), (k, name, call)
    batch.close()


def add_extras(sim, pol, wx, wy, downsample):
    """A Drude rectangle (E_z), DFT boxes with and without a stride, and probes near the window edges."""
    from opensol_amd import DrudePole
    if pol == 'ez':
        sim.add_drude_rectangle(0.3 * wx * DX, 0.1 * wy * DX, 0.8 * wx * DX, 0.9 * wy * DX,
                                DrudePole(omega_p=1.5e15, gamma=1e14, eps_inf=4.0))
    sim.add_dft_monitor(0.5 * DX, 0.5 * DX, (wx - 0.5) * DX, (wy - 0.5) * DX, wavelengths=[550e-9, 700e-9],
                        downsample=downsample)
    sim.add_dft_monitor(0.2 * wx * DX, 0.3 * wy * DX, 0.7 * wx * DX, 0.8 * wy * DX, wavelengths=[600e-9])
    rng = np.random.default_rng([wx, wy])
    components = ('ez', 'hx', 'hy') if pol == 'ez' else ('hz', 'ex', 'ey')
    spots = [(0, 0), (wx - 1, wy - 1)] + [(rng.integers(wx), rng.integers(wy)) for _ in range(9)]
    for k, (i, j) in enumerate(spots):
        sim.add_field_probe((i + 0.5) * DX, (j + 0.5) * DX, field_component=components[k % 3])


@pytest.mark.parametrize('pol', ['ez', 'hz'])
@pytest.mark.parametrize('nx,ny', [(34, 64), (61, 37), (129, 130), (300, 257), (611, 523)])
@pytest.mark.parametrize('boundaries,media', [('pml', 'plain'), ('periodic_y', 'lossy'), ('periodic_x', 'plain'),
                                              ('periodic', 'pec')])
@pytest.mark.parametrize('graph_steps', [0, 9])
def test_multi_step_with_pole_regions_and_probes(gpu, pol, nx, ny, boundaries, media, graph_steps):
    def make(graph):
        return build(pol, nx, ny, boundaries, media, graph,
                     extras=lambda sim, wx, wy: add_extras(sim, pol, wx, wy, 3 if nx % 2 else 1))
    multi, single = make(graph_steps), make(0)
    total = 0
    for steps in (1, 2, 7, 20, 33):
        multi.engine.step(steps)
        single.engine.step_timed(steps)
        total += steps
        a, b = arrays(multi, total), arrays(single, total)
        for sim, out in ((multi, a), (single, b)):
            out.update({f'dft {k}': acc for k, acc in enumerate(sim.engine.dft_accumulators)})
            out.update({f'current {k}': entry['states'][0] for k, entry in enumerate(sim.engine.poles)})
            out['probes'] = sim.engine.probes.samples[:total]
        for name in a:
            assert bool((a[name] == b[name]).all()), (name, total, int((a[name] != b[name]).sum()))
    assert all(bool((acc != 0).any()) for acc in multi.engine.dft_accumulators)


@pytest.mark.parametrize('pol', ['ez', 'hz'])
def test_calls_of_one_and_two_steps_of_a_large_grid(gpu, pol):
    """One- and two-step calls of a large grid take other kernels than longer ones: the state passes between them."""
    multi, single = (build(pol, 2051, 2046, 'pml', 'plain',
                           extras=lambda sim, wx, wy: add_extras(sim, pol, wx, wy, 4)) for _ in range(2))
    total = 0
    for steps in (1, 3, 2, 7, 1):
        multi.engine.step(steps)
        single.engine.step_timed(steps)
        total += steps
        a, b = arrays(multi, total), arrays(single, total)
        for sim, out in ((multi, a), (single, b)):
            out.update({f'current {k}': entry['states'][0] for k, entry in enumerate(sim.engine.poles)})
            out['probes'] = sim.engine.probes.samples[:total]
        for name in a:
            assert bool((a[name] == b[name]).all()), (name, total)


def overflowed(sim, nx, ny):
    """Infinities and values near the largest float in and beside the layers, the grid's last rows and the bulk."""
    torch = sim.engine.torch
    fields = sim.engine.fields[0]
    huge = 3.0e38
    for c in range(3):
        for i, j, v in ((0, 3, float('inf')), (nx - 1, ny // 3, -float('inf')), (nx // 3, ny - 1, float('inf')),
                        (nx // 2, 0, -huge), (nx // 2 + 3, ny // 2, huge), (nx // 2 + 3, ny // 2 + 1, -huge),
                        (NPML + 2, NPML + 2, float('inf')), (nx - NPML - 3, ny - NPML - 4, huge),
                        (nx - NPML - 3, ny - NPML - 3, -huge)):
            fields[c, min(max(i + c, 0), nx - 1), min(max(j + c, 0), ny - 1)] = v
    assert torch.isinf(fields).any()


@pytest.mark.parametrize('pol', ['ez', 'hz'])
@pytest.mark.parametrize('nx,ny', [(34, 64), (129, 130), (300, 257)])
@pytest.mark.parametrize('boundaries,media', [('pml', 'plain'), ('periodic_y', 'lossy'), ('periodic_x', 'plain'),
                                              ('pml', 'pec')])
@pytest.mark.parametrize('extras', [False, True])
def test_overflowed_fields_stay_what_single_steps_make_of_them(gpu, pol, nx, ny, boundaries, media, extras):
    """An infinity spreads and cancels to NaN in the same cells, however many steps a launch takes."""
    def make():
        return build(pol, nx, ny, boundaries, media,
                     extras=(lambda sim, wx, wy: add_extras(sim, pol, wx, wy, 2)) if extras else None)
    multi, single = make(), make()
    for sim in (multi, single):
        overflowed(sim, nx, ny)
    total = 0
    for steps in (1, 2, 5, 9):
        multi.engine.step(steps)
        single.engine.step_timed(steps)
        total += steps
        a, b = arrays(multi, total), arrays(single, total)
        for name in a:
            same = (a[name] == b[name]) | (a[name].isnan() & b[name].isnan()) if a[name].is_floating_point() else \
                a[name] == b[name]
            assert bool(same.all()), (name, total, int((~same).sum()))
    assert bool(arrays(multi, total)['fields'].isnan().any())


def test_infinite_source_value_stays_within_its_span(gpu):
    """A source table that holds an infinity adds it to the cells of its span and leaves the others of its line alone."""
    def line(sim, wx, wy):
        sim.add_line_source(axis='y', position=0.5 * wx * DX, wavelength=600e-9, span=(0.3 * wy * DX, 0.6 * wy * DX))
    sims = [build('ez', 129, 130, 'pml', 'plain', extras=line) for _ in range(2)]
    for sim in sims:
        sim.engine.waves[-1][2] = float('inf')
    sims[0].engine.step(3)
    sims[1].engine.step_timed(3)
    a, b = (arrays(sim, 3)['fields'] for sim in sims)
    assert bool(((a == b) | (a.isnan() & b.isnan())).all()) and bool(a.isinf().any())


@pytest.mark.parametrize('pol', ['ez', 'hz'])
@pytest.mark.parametrize('downsample,wavelengths', [(1, 1), (1, 2), (1, 8), (2, 24), (1, 100)])
def test_multi_step_with_dense_regions(gpu, pol, downsample, wavelengths):
    """DFT regions over the whole grid, from a small share of a step to all of it: the windows and kernels chosen for them
    take the same samples."""
    def region(sim, wx, wy):
        sim.add_dft_monitor(0.5 * DX, 0.5 * DX, (wx - 0.5) * DX, (wy - 0.5) * DX, downsample=downsample,
                            wavelengths=list(np.linspace(500e-9, 800e-9, wavelengths)))
    multi, single = (build(pol, 611, 523, 'pml', 'plain', extras=region) for _ in range(2))
    total = 0
    for steps in (2, 7, 20):
        multi.engine.step(steps)
        single.engine.step_timed(steps)
        total += steps
    a, b = arrays(multi, total), arrays(single, total)
    a['dft'], b['dft'] = (sim.engine.dft_accumulators[0] for sim in (multi, single))
    for name in a:
        assert bool((a[name] == b[name]).all()), (name, total)
    assert bool((a['dft'] != 0).any())


def test_small_batches_take_several_steps_a_launch(gpu):
    """Two small members in calls of 25 steps: several steps a launch, unless the batch is told to take one."""
    from opensol_amd.batch import Batch2D
    members, singles = ([build('ez', 84, 69, 'pml', 'plain'), build('hz', 61, 73, 'pml', 'plain')] for _ in range(2))
    paced, free = Batch2D(singles), Batch2D(members)
    paced.multi_step = False
    for batch, several in ((paced, False), (free, True)):
        for _ in range(3):
            batch.prepare(25)
            assert (batch.lib.yee_steps_per_launch(batch._ctx, 25) > 1) == several
            batch.launch()
    for a, b in zip(members, singles):
        got, expected = arrays(a, 75), arrays(b, 75)
        for name in got:
            assert bool((got[name] == expected[name]).all()), name
    paced.close()
    free.close()


@pytest.mark.parametrize('pol', ['ez', 'hz'])
@pytest.mark.parametrize('axis', ['x', 'y'])
def test_periodic_axis_with_layers(gpu, pol, axis):
    """A descriptor may wrap an axis that has CPML rows, which no model does: both launch forms step it alike."""
    import ctypes
    from opensol_amd import _lib
    sims = [build(pol, 129, 130, 'pml', 'lossy') for _ in range(2)]
    for sim in sims:
        d = sim.engine.descriptor()
        setattr(d, f'periodic_{axis}', 1)
        _lib.check(sim.engine.lib.yee2d_update(sim.engine._ctx, ctypes.byref(d)), 'yee2d_update')
    sims[0].engine.step(20)
    sims[1].engine.step_timed(20)
    a, b = (arrays(sim, 20) for sim in sims)
    for name in a:
        assert bool((a[name] == b[name]).all()), name


@pytest.mark.parametrize('pol', ['ez', 'hz'])
@pytest.mark.parametrize('axis', ['x', 'y'])
def test_uneven_spacings_without_layers(gpu, pol, axis):
    """A descriptor whose layer bounds leave no bulk along an axis takes its spacings from the arrays, with or without CPML."""
    import ctypes
    from opensol_amd import _lib
    sims = [build(pol, 129, 130, 'periodic', 'lossy') for _ in range(2)]
    for sim in sims:
        d = sim.engine.descriptor()
        n = getattr(d, f'n{axis}')
        torch = sim.engine.torch
        stretch = torch.linspace(0.7, 1.0, n, device=sim.engine.device)
        sim.spacings = [t * stretch for t in sim.engine.inv[0 if axis == 'x' else 2:][:2]]
        for name, t in zip(('e', 'h'), sim.spacings):
            setattr(d, f'inv_d{axis}_{name}', t.data_ptr())
        setattr(d, f'layer_{axis}_lo', n)
        _lib.check(sim.engine.lib.yee2d_update(sim.engine._ctx, ctypes.byref(d)), 'yee2d_update')
    sims[0].engine.step(20)
    sims[1].engine.step_timed(20)
    a, b = (arrays(sim, 20) for sim in sims)
    for name in a:
        assert bool((a[name] == b[name]).all()), name
