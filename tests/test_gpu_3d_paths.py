"""The fused 3D step kernel against the two-launch one (H, then E): an instance alone is below the size from which steps are
fused, in a batch with a large one it is above it. Every field, psi array, pole state, accumulator and probe sample is equal
bit for bit, from random fields, at sizes around the fused kernel's tiles (64 z cells x 14 rows)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DX = 25e-9
ALL = tuple(f'{a}_{e}' for a in 'xyz' for e in ('lo', 'hi'))


def periodic(axes):
    return {f'{a}_{e}': 'periodic' for a in axes for e in ('lo', 'hi')}


# (grid cells x, y, z, npml, faces, planes per tile in the batch)
CASES = [((20, 13, 63), 2, None, 0), ((21, 14, 64), 3, None, 4), ((40, 15, 65), 2, None, 7), ((24, 44, 200), 3, None, 3),
         ((9, 29, 66), 0, periodic('xyz'), 2), ((17, 5, 3), 0, periodic('xyz'), 40), ((30, 28, 129), 4, periodic('x'), 5),
         ((12, 43, 130), 3, periodic('y'), 1), ((26, 33, 128), 3, periodic('z'), 6),
         ((25, 30, 140), 4, {'x_lo': 'symmetric', 'y_hi': 'antisymmetric', 'z_lo': 'symmetric'}, 5),
         ((25, 30, 70), 4, {'x_hi': 'symmetric', 'y_lo': 'symmetric', 'z_hi': 'antisymmetric'}, 0)]


def build(shape, npml, faces, seed, extras=True):
    from opensol_amd import Simulation3D
    from opensol_amd.dispersion import DrudePole, LorentzPole
    faces = faces or {}

    def pads(axis):   # cells beyond the window: CPML rows, one ghost cell on a mirror face
        return sum({'periodic': 0, 'symmetric': 1, 'antisymmetric': 1}.get(faces.get(f'{axis}_{e}'), npml)
                   for e in ('lo', 'hi'))
    size = tuple((n - pads(a)) * DX for n, a in zip(shape, 'xyz'))
    sim = Simulation3D(*size, DX, npml=npml, boundaries=faces)
    assert sim.model.shape == shape
    rng = np.random.default_rng(seed)
    for _ in range(5):
        lo = rng.uniform(-0.2, 1.0, 3) * np.array(size)
        hi = lo + rng.uniform(0.1, 0.6, 3) * np.array(size)
        sim.add_dielectric_box(tuple(lo), tuple(hi), rng.uniform(1, 9), 2e4 if rng.random() < 0.3 else 0.0)
    sim.add_pec_box(tuple(0.6 * s for s in size), tuple(0.75 * s for s in size))
    if extras:
        for orientation, at in (('z', 0.5), ('x', 0.25)):
            sim.add_dipole(*(at * s for s in size), orientation=orientation, dipole_moment=3e-18, wavelength=600e-9,
                           bandwidth=0.5)
        sim.add_flux_plane('x', 0.5 * size[0], wavelengths=[600e-9])
        sim.add_field_probe(*(0.4 * s for s in size), component='hy')
    if extras == 'poles':
        window, mask = tuple(slice(0, n) for n in shape), np.zeros(shape, bool)
        mask[2:7, 1:, :-1] = True
        sim.add_dispersive(DrudePole(2e15, 1e14), window, mask)
        sim.add_dispersive(LorentzPole(1.5, 3e15, 2e14), window, mask)
    sim.finalize()
    torch = sim.engine.torch
    generator = torch.Generator().manual_seed(seed)
    fields = sim.engine.fields[0]
    for c in range(6):
        fields[c].copy_(torch.randn(shape, generator=generator) * (1.0 if c < 3 else 1 / 376.7))
    return sim


def state(sim, n):
    e = sim.engine
    out = {'fields': e.fields[n & 1]}
    for name, axis in e.cpml.items():
        if axis is not None:
            out[f'psi_e {name}'], out[f'psi_h {name}'] = axis['psi_e'], axis['psi_h'][n & 1]
    out.update({f'acc {k} {q}': a for k, m in enumerate(e.accumulators) for q, a in enumerate(m)})
    out.update({f'pole {k} {q}': a for k, p in enumerate(e.poles) for q, a in enumerate(p['states'])})
    out['probes'] = e.probes.samples[:n]
    return out


@pytest.mark.parametrize('shape,npml,faces,planes', CASES)
def test_fused_step_matches_the_two_launches(gpu, shape, npml, faces, planes):
    from opensol_amd.batch import Batch3D
    extras = 'poles' if min(shape) > 12 else True
    alone, member = (build(shape, npml, faces, 7, extras) for _ in range(2))
    large = build((130, 250, 260), 3, None, 8, extras=False)   # 8.45M cells
    batch = Batch3D([member, large], planes_per_tile=planes)
    total = 0
    for steps in (1, 4, 5):
        alone.engine.step(steps)
        batch.run([steps, 1])
        total += steps
        a, b = state(alone, total), state(member, total)
        for name in a:
            assert bool((a[name] == b[name]).all()), (name, total, int((a[name] != b[name]).sum()))
    batch.close()
    for sim in (alone, member, large):
        sim.close()
