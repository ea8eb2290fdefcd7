"""Energy reductions and the distribution-array copies at the edges of their
launches: boxes smaller than the enstrophy stencil, rows and chunks (2048 nodes)
with remainders, with and without solid nodes, and arrays around the 1024
elements of a copy workgroup."""
import numpy as np
import pytest
import torch

import oracle
import virtualfluids_amd as vfx
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solid_share", [0.0, 0.03])
@pytest.mark.parametrize("dims", [(3, 5, 4), (1, 2, 70), (17, 9, 12), (65, 33, 8), (41, 37, 25)])
def test_energies_match_the_oracle(cuda, dims, solid_share):
    """Sums of positive terms in FP64: 1e-12 of the sum covers the rounding of
    n <= 37925 additions and of the stencil (as tests of the same kernels do).
    The largest box has 19 chunks of 2048 nodes: two per XCD and three after
    them, so that the chunks' order is not the blocks'."""
    print(f"[energies {dims} {solid_share}]", flush=True)
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    solid = rng.random(n) < solid_share if solid_share else None
    F0 = oracle.init_field(*cases.random_flow(dims, seed=n))
    lat = vfx.Lattice(dims, storage="fp64", omega=1.8, solid=solid)
    lat.write_populations(F0)
    if solid is not None:
        F0[solid] = 0.0
    for name, f in (("ke", lat.kinetic_energy), ("enstrophy", lat.enstrophy)):
        got = f().cpu().numpy()
        ref = np.asarray(oracle.energy(F0, dims, enstrophy=name == "enstrophy",
                                       solid=np.zeros(n, bool) if solid is None else solid))
        assert got[1] == ref[1]
        assert abs(got[0] - ref[0]) <= 1e-12 * abs(ref[0]) + 1e-30


@pytest.mark.parametrize("even", [True, False])
@pytest.mark.parametrize("storage", ["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("dims", [(1, 1, 1), (31, 33, 1), (32, 32, 1), (41, 25, 1), (41, 25, 3)])
def test_distribution_array_round_trip(cuda, dims, storage, even):
    print(f"[array {dims} {storage} {even}]", flush=True)
    n = int(np.prod(dims))
    a = vfx.Lattice(dims, storage=storage, omega=1.8,
                    reference_velocity=(0.03, 0.01, -0.02) if storage == "fp16" else (0.0, 0.0, 0.0))
    a.init_equilibrium(*cases.random_flow(dims, seed=n), even=even)
    real = torch.float64 if storage == "fp64" else torch.float32
    x = a.export_distributions(even, real)
    if storage != "fp16":
        assert torch.equal(x, a.f)
    pops = a.read_populations(even).cpu().numpy()
    planes = x.double().cpu().numpy().reshape(27, n)
    k = np.arange(n)
    for d in range(27):
        xx = (k % dims[0] + (vfx.CX[d] < 0)) % dims[0]
        yy = (k // dims[0] % dims[1] + (vfx.CY[d] < 0)) % dims[1]
        zz = (k // (dims[0] * dims[1]) + (vfx.CZ[d] < 0)) % dims[2]
        at = xx + dims[0] * (yy + dims[1] * zz)
        assert np.array_equal(planes[d if even else vfx.INV[d], at], pops[:, d])
    b = vfx.Lattice(dims, storage=storage, omega=1.8, reference_velocity=a.reference_velocity)
    b.import_distributions(x, even)
    if storage == "fp16":
        # the decoded value carries the FP32 rounding of h + offset (offset below 300 units of h at this
        # velocity), so a small h may come back as its neighbour: one step of the half plus that rounding
        h = a.f.double()
        assert bool(((b.f.double() - h).abs() <= 2.0 ** -10 * h.abs() + 2.0 ** -23 * 300.0).all())
    else:
        assert torch.equal(a.f, b.f)
    y = x.clone()
    y[0] = float("nan")
    b.import_distributions(y, even)
    assert float(b.export_distributions(even, real)[0]) == 0.0
