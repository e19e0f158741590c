"""Which calls take several steps a launch, as the library answers it (yee_steps_per_launch) for descriptors that are never
stepped: their device pointers are stand-ins."""
import ctypes

import pytest

from opensol_amd import _lib

POINTER = 1 << 20


@pytest.fixture(scope='module')
def lib():
    return _lib.load()


def descriptor(nx, ny, pol='ez'):
    d = _lib.Desc2DC()
    d.nx, d.ny, d.pitch = nx, ny, (ny + 3) // 4 * 4
    d.polarization = _lib.YEE_EZ if pol == 'ez' else _lib.YEE_HZ
    for s in range(2):
        for c in range(3):
            d.field[s][c] = POINTER
    d.material = d.table = d.table2 = d.inv_dx_e = d.inv_dx_h = d.inv_dy_e = d.inv_dy_h = d.clock = POINTER
    d.n_materials, d.sample_interval, d.step_limit = 3, 1, _lib.INT64_MAX
    d.layer_x_hi, d.layer_y_hi = nx, ny
    return d


def layers(d, axis, rows):
    c = d.cpml[axis]
    c.n_rows = rows
    for name in ('row_e', 'row_h', 'b_e', 'g_e', 'b_h', 'g_h'):
        setattr(c, name, POINTER)
    for s in range(2):
        c.psi_e[s] = c.psi_h[s] = POINTER


def steps_per_launch(lib, d, n, multi=None):
    ctx = _lib.c_ptr()
    _lib.check(lib.yee2d_create(ctypes.byref(d), ctypes.byref(ctx)), 'yee2d_create')
    try:
        if multi is not None:
            _lib.check(lib.yee_set_multi_step(ctx, multi), 'yee_set_multi_step')
        return lib.yee_steps_per_launch(ctx, n)
    finally:
        lib.yee_destroy(ctx)


def test_calls_take_several_steps_a_launch_unless_told_otherwise(lib):
    d = descriptor(300, 257)
    assert steps_per_launch(lib, d, 100) > 3
    assert steps_per_launch(lib, d, 1) == 1 and steps_per_launch(lib, d, 0) == 0
    assert steps_per_launch(lib, d, 100, multi=0) == 1 and steps_per_launch(lib, d, 100, multi=1) > 3
    d.step_limit = 50
    assert steps_per_launch(lib, d, 100) == 1
    assert lib.yee_steps_per_launch(None, 5) == 0


def test_layers_of_a_periodic_x_axis_are_stepped_one_launch_at_a_time(lib):
    """The windows hold the x layers' rows by the grid's own index, so they do not follow a wrap around such an axis."""
    d = descriptor(300, 257)
    layers(d, 0, 16)
    assert steps_per_launch(lib, d, 100) > 3
    d.periodic_x = 1
    assert steps_per_launch(lib, d, 100) == 1
    d.periodic_x, d.periodic_y = 0, 1
    layers(d, 1, 16)
    assert steps_per_launch(lib, d, 100) > 3


def test_spacings_of_layer_bounds_without_cpml_are_stepped_one_launch_at_a_time(lib):
    d = descriptor(300, 257)
    d.layer_y_lo = 257
    assert steps_per_launch(lib, d, 100) > 3
    for lo, hi in ((300, 300), (0, 0), (5, 300)):
        d.layer_x_lo, d.layer_x_hi = lo, hi
        assert steps_per_launch(lib, d, 100) == 1
    layers(d, 0, 16)
    assert steps_per_launch(lib, d, 100) > 3


@pytest.mark.parametrize('nx,ny,several', [(2, 2_000_000_000, False), (2, 300_000_000, True), (100_000, 100_000, True)])
@pytest.mark.parametrize('pol', ['ez', 'hz'])
def test_grids_with_more_windows_than_a_launch_holds_step_one_launch_at_a_time(lib, pol, nx, ny, several):
    """A launch has fewer than 2^32 threads, 512 a window of at most 64 columns."""
    assert (steps_per_launch(lib, descriptor(nx, ny, pol), 100) > 1) == several


def test_a_server_paces_small_members_only_when_it_preempts():
    from opensol_amd.serve import FDTDServer, Job
    small = [Job(build=None, steps=10, arrival=0.0, cells=5000) for _ in range(2)]
    for job in small:
        job.sim = type('Sim', (), {'model': type('Model', (), {'shape': (50, 100)})})
    assert FDTDServer(chunk_steps=25, preempt_after=0.0)._paced(small)
    assert not FDTDServer(chunk_steps=25)._paced(small)
    assert not FDTDServer(chunk_steps=32, preempt_after=0.0)._paced(small)
    assert not FDTDServer(chunk_steps=25, preempt_after=0.0)._paced(small * 2)
