"""The autotuner chooses options for the kernels that read them: 2D shapes with one step a launch, 3D planes for the step form
of the member, left behind in a batch of the other form."""
import pytest

from opensol_amd import autotune


class _Model:
    def __init__(self, shape, polarization=None):
        self.shape = shape
        self.polarization = polarization


def test_step_form_is_part_of_a_3d_class():
    assert autotune.tuned_key('batch', _Model((130, 130, 130))) == 'batch:3d:8x8x8:split'
    assert autotune.tuned_key('batch', _Model((250, 250, 250))) == 'batch:3d:8x8x8:fused'
    assert autotune.tuned_key('single', _Model((100, 100, 100))) == 'single:3d:7x7x7:split'
    assert autotune.tuned_key('batch', _Model((300, 700), 'ez'), 4) == 'batch:ez:9x10:lanes4'
    assert autotune.tuned_key('single', _Model((300, 700), 'hz')) == 'single:hz:9x10'


@pytest.mark.gpu
def test_2d_shapes_are_timed_with_one_step_a_launch(gpu, monkeypatch):
    from opensol_amd import Simulation
    seen = []
    monkeypatch.setattr(autotune, '_elapsed_ms', lambda run, steps, torch: seen.append(
        run.__self__.lib.yee_steps_per_launch(run.__self__._ctx, steps)) or float(len(seen)))

    def batch_ms(batch, steps, torch):
        batch.prepare(steps)
        seen.append(batch.lib.yee_steps_per_launch(batch._ctx, steps))
        return float(len(seen))
    monkeypatch.setattr(autotune, '_batch_ms', batch_ms)
    for tune in (autotune.tune, autotune.tune_batch_member):
        sim = Simulation(5e-6, 4e-6, 25e-9, npml=8, polarization='ez')
        sim.add_line_source(axis='y', position=1e-6, wavelength=600e-9)
        tune(sim, use_cache=False, cache=autotune.TuneCache('/nonexistent/tune.json'))
        sim.finalize()
        assert sim.engine.lib.yee_steps_per_launch(sim.engine._ctx, 10) > 1
        sim.close()
    assert len(seen) == len(autotune.CANDIDATES_2D) + len(autotune.BATCH_ROWS_2D) and set(seen) == {1}


@pytest.mark.gpu
def test_tuned_planes_stay_with_their_step_form(gpu, monkeypatch):
    from opensol_amd import Simulation3D
    from opensol_amd.batch import Batch3D
    dx, sims = 25e-9, []
    for cells in ((24, 20, 28), (24, 20, 28), (130, 250, 260)):
        sim = Simulation3D(*(n * dx for n in cells), dx, npml=4)
        sim.add_dipole(*(0.5 * n * dx for n in cells), wavelength=600e-9)
        sims.append(sim)
    small, chosen, large = sims
    cache = autotune.TuneCache('/nonexistent/tune.json')
    monkeypatch.setattr(autotune, '_batch_ms', lambda batch, steps, torch: 1.0 / (1 + batch.simulations[0].engine.planes_per_tile))
    options, timings = autotune.tune_batch_member(small, use_cache=False, cache=cache)
    assert options == {'planes_per_tile': max(autotune.BATCH_PLANES_3D)} and len(timings) == len(autotune.BATCH_PLANES_3D)
    chosen._engine_options['planes_per_tile'] = 3   # the caller's own number
    planes = []

    def create(self, descs, *args):
        planes.append([d.planes_per_tile for d in descs])
        return self.lib.yee3d_batch_create(descs, *args)
    monkeypatch.setattr(Batch3D, '_create', create)
    for members in ([small, chosen], [small, chosen, large]):
        batch = Batch3D(members)
        batch.run(2)
        batch.close()
    assert planes == [[max(autotune.BATCH_PLANES_3D), 3], [0, 3, 0]]
    for sim in sims:
        sim.close()
