"""Rows of 256 in one block whose number squared leaves 32 bits: the chunk list's
cuts take 64 (20 million particles in 64 cells; with 32 the last 23,150 of 78,125
chunks would hold other chunks' particles)."""
import pytest
import torch

from femflow_amd.engine import Engine, MaterialSpec, SceneSpec


@pytest.mark.gpu
def test_every_particle_of_a_dense_block_is_taken_once(gpu):
    """Particles at rest, unstrained, one substep: every particle has the speed
    that gravity gives in dt (one that no chunk held would keep none), and the
    grid holds the particles' mass (one in two chunks would count twice), to the
    FP32 rounding of its 78,125 chunks' sums."""
    n, dt = 20_000_000, 1e-4
    g = torch.Generator(device=gpu).manual_seed(1)
    x = (8.75 + 3.2 * torch.rand(n, 3, generator=g, device=gpu)) / 32  # bases 8..11: one block
    zero = lambda *s: torch.zeros(*s, device=gpu)  # noqa: E731
    full = lambda a: torch.full((n,), a, device=gpu)  # noqa: E731
    F = torch.eye(3, device=gpu).repeat(n, 1, 1)
    eng = Engine([SceneSpec(res=32, dt=dt, gravity=-9.8, volume=1e-9)], [MaterialSpec("elastic")], n_max=n)
    eng.tune(chunk=256)
    eng.upload(x, zero(n, 3), F, zero(n, 3, 3), full(1.0), full(2.0 ** -20), full(1.0), full(1.0))
    sums = torch.zeros(1, 8, dtype=torch.float64, device=gpu)
    eng.run(1, sums=sums)
    v = zero(n, 3)
    eng.download(torch.empty_like(x), v, F, zero(n, 3, 3), full(1.0))
    assert abs(float(sums[0, 0]) - n * 2.0 ** -20) <= 78_125 * 2.0 ** -24 * n * 2.0 ** -20
    assert float((v - torch.tensor([0.0, -9.8 * dt, 0.0], device=gpu)).abs().max()) <= 1e-5 * 9.8 * dt
    eng.close()
