"""The launch forms at the ends of what they hold: as many materials as the windows of several 2D steps keep in LDS and one
more, as many as the fused 3D step keeps and one more, 64 probes and one more. Each against the other launch form, bit for
bit, with the last ids of the table in the grid."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DX, NPML = 25e-9, 8


def grid_2d(pol, materials, media, probes=0):
    from opensol_amd import Simulation
    wx, wy = 284, 241
    sim = Simulation(wx * DX, wy * DX, DX, npml=NPML, polarization=pol)
    rng = np.random.default_rng(materials)
    for k in range(materials - 1):
        i, j = rng.integers(0, wx - 9), rng.integers(0, wy - 9)
        sim.add_dielectric_rectangle(i * DX, j * DX, (i + 9) * DX, (j + 9) * DX, eps_r=1.5 + 0.01 * k,
                                     sigma_e=1e3 + k if media == 'lossy' else 0.0)
    sim.add_line_source(axis='y', position=0.3 * wx * DX, wavelength=600e-9, waveform='ricker')
    for _ in range(probes):
        sim.add_field_probe((rng.integers(wx) + 0.5) * DX, (rng.integers(wy) + 0.5) * DX)
    sim.finalize()
    assert len(sim.model.materials.materials) == materials and sim.model.materials.ids.max() == materials - 1
    generator = sim.engine.torch.Generator().manual_seed(materials)
    fields = sim.engine.fields[0, :, :, :sim.model.ny]
    fields.copy_(sim.engine.torch.randn(fields.shape, generator=generator))
    return sim


@pytest.mark.parametrize('pol,materials', [('ez', 1023), ('ez', 1024), ('hz', 511), ('hz', 512)])
@pytest.mark.parametrize('media', ['plain', 'lossy'])
def test_materials_of_the_windows(gpu, pol, materials, media):
    multi, single = (grid_2d(pol, materials, media) for _ in range(2))
    assert (multi.engine.steps_per_launch(20) > 1) == (materials in (1023, 511))
    multi.engine.step(20)
    single.engine.step_timed(20)
    assert bool((multi.engine.fields[0] == single.engine.fields[0]).all())


@pytest.mark.parametrize('probes', [64, 65])
def test_probes_of_the_windows(gpu, probes):
    multi, single = (grid_2d('ez', 9, 'plain', probes) for _ in range(2))
    assert (multi.engine.steps_per_launch(20) > 1) == (probes == 64)
    multi.engine.step(20)
    single.engine.step_timed(20)
    for a, b in ((multi.engine.fields[0], single.engine.fields[0]),
                 (multi.engine.probes.samples[:20], single.engine.probes.samples[:20])):
        assert bool((a == b).all())


def grid_3d(shape, materials):
    from opensol_amd import Simulation3D
    npml = 3
    size = np.array([n - 2 * npml for n in shape])
    sim = Simulation3D(*(size * DX), DX, npml=npml)
    rng = np.random.default_rng(materials)
    for k in range(materials - 1):
        lo = rng.integers(0, size - 5)
        sim.add_dielectric_box(tuple(lo * DX), tuple((lo + 5) * DX), 1.5 + 0.01 * k, 1e3 + k)
    sim.finalize()
    assert len(sim.model.materials.materials) == materials
    generator = sim.engine.torch.Generator().manual_seed(materials)
    sim.engine.fields[0].copy_(sim.engine.torch.randn(sim.engine.fields[0].shape, generator=generator))
    return sim


@pytest.mark.parametrize('materials', [512, 513])
def test_materials_of_the_fused_3d_step(gpu, materials):
    from opensol_amd.batch import Batch3D
    alone, member = (grid_3d((30, 31, 70), materials) for _ in range(2))
    large = grid_3d((130, 250, 260), 2)   # 8.45M cells: the batch steps in fused launches, the one alone in two
    assert large.engine.lib.yee3d_fused(8_450_000) == 1 and large.engine.lib.yee3d_fused(30 * 31 * 70) == 0
    batch = Batch3D([member, large])
    alone.engine.step(5)
    batch.run([5, 1])
    assert bool((alone.engine.fields[1] == member.engine.fields[1]).all())
    batch.close()
    for sim in (alone, member, large):
        sim.close()
