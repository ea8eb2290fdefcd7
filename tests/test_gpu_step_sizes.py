"""The structured step on boxes whose rows, slabs and node count do not fit its
tiles or wavefronts, against the oracle: FP64 reproduces it bit for bit.
The sizes sit at the edges of the flat node mapping (one node in a direction,
rows of one node more or less than a wavefront, a last tile of one node)."""
import numpy as np
import pytest
import torch

import oracle
import virtualfluids_amd as vfx
from tests import cases

pytestmark = pytest.mark.gpu

DIMS = [(1, 5, 7), (5, 1, 7), (5, 7, 1), (63, 3, 2), (64, 3, 2), (65, 3, 2), (257, 2, 2), (1, 1, 257), (33, 31, 9)]


@pytest.mark.parametrize("collision", ["k17", "bgk"])
@pytest.mark.parametrize("dims", DIMS)
def test_box_sizes_bitwise_in_fp64(cuda, dims, collision):
    print(f"[step {dims} {collision}]", flush=True)
    F0 = oracle.init_field(*cases.random_flow(dims, seed=sum(dims)))
    lat = vfx.Lattice(dims, storage="fp64", omega=1.85)
    lat.write_populations(F0)
    st = vfx.Stepper(lat, collision)
    st.step(3)
    ref = oracle.run(F0, dims, 3, 1.85, collision=collision)
    assert np.array_equal(st.populations().cpu().numpy(), ref)


@pytest.mark.parametrize("model", ["smagorinsky", "qr", "amd"])
@pytest.mark.parametrize("sparse", [False, True])
def test_fp16_models_reduced_form_equals_the_reference_order(cuda, model, sparse):
    """FP16 storage runs the reduced-operation K17 with the node's own rates,
    variant="plain" the reference order: one step differs by the FP32 rounding
    of ~1500 operations (1e-5 of the largest population, generous) plus one unit
    of the half it is stored in (2^-10 of the population itself).  The eddy
    viscosity is compared with FP64's from the same populations: the reduced
    form is no further off than the reference order."""
    print(f"[fp16 {model} {sparse}]", flush=True)
    dims = (37, 11, 8)
    n = int(np.prod(dims))
    fields = cases.random_flow(dims, seed=4)
    nut = 1e-3 * (1.0 + np.sin(np.arange(n)))
    out = []
    for storage, variant in (("fp16", "default"), ("fp16", "plain"), ("fp64", "default")):
        kw = dict(storage=storage, omega=1.97, turbulence=model, sgs_constant=0.2, variant=variant)
        if sparse:
            k = np.arange(n)
            x, y, z = k % dims[0], k // dims[0] % dims[1], k // (dims[0] * dims[1])

            def at(a, b, c):
                return (a % dims[0] + dims[0] * (b % dims[1] + dims[1] * (c % dims[2]))).astype(np.uint32)
            lat = vfx.Lattice(neighbors=(at(x + 1, y, z), at(x, y + 1, z), at(x, y, z + 1)),
                              node_types=np.full(n, 19, np.uint32), neighbor_inverse=at(x - 1, y - 1, z - 1), **kw)
        else:
            lat = vfx.Lattice(dims, **kw)
        if storage == "fp16":
            lat.init_equilibrium(*fields)
            start = lat.read_populations()
        else:
            lat.write_populations(start)
        lat.nut.copy_(torch.from_numpy(nut).to(lat.nut.dtype))
        vfx.Stepper(lat, "k17").step(1)
        out.append((lat.f.double().cpu().numpy().reshape(27, n), lat.nut.double().cpu().numpy()))
    (a, va), (b, vb), (_, v) = out
    assert np.all(np.abs(a - b) <= 1e-5 * np.abs(b).max(axis=1, keepdims=True) + 2.0 ** -10 * np.abs(b))
    assert np.linalg.norm(va - v) <= np.linalg.norm(vb - v)
    assert not np.array_equal(a, b)  # the two forms did run


@pytest.mark.parametrize("model", ["smagorinsky", "qr", "amd"])
@pytest.mark.parametrize("dims,body_force", [((37, 11, 8), False), ((65, 16, 9), False), ((37, 11, 8), True)])
def test_fp16_models_write_the_reference_orders_density_and_velocity(cuda, model, dims, body_force):
    """The 32-bit fields the collision writes, and the viscosity the AMD kernel
    forms from them, are the same bits in the default and the "plain" variant."""
    print(f"[fp16 fields {model} {dims} {body_force}]", flush=True)
    n = int(np.prod(dims))
    nut = torch.from_numpy(1e-3 * (1.0 + np.sin(np.arange(n)))).float()
    force = 1e-4 * np.sin(np.arange(n)), 1e-4, -1e-4 * np.cos(np.arange(n))
    out = []
    for variant in ("default", "plain"):
        lat = vfx.Lattice(dims, storage="fp16", omega=1.95, turbulence=model, sgs_constant=0.2, variant=variant)
        lat.init_equilibrium(*cases.random_flow(dims, seed=9))
        lat.nut.copy_(nut)
        if body_force:
            lat.set_body_force(*force, forces=(1e-5, 0.0, 0.0))
        lat.collide_stream("k17", True, write_macro=True, apply_body_force=body_force)
        fields = list(lat.macro)
        if model == "amd":
            lat.turbulent_viscosity_amd()
            fields.append(lat.nut)
        out.append(fields)
        if variant == "default" and model != "amd":
            # writing the fields changes no population
            c = vfx.Lattice(dims, storage="fp16", omega=1.95, turbulence=model, sgs_constant=0.2)
            c.init_equilibrium(*cases.random_flow(dims, seed=9))
            c.nut.copy_(nut)
            if body_force:
                c.set_body_force(*force, forces=(1e-5, 0.0, 0.0))
            c.collide_stream("k17", True, apply_body_force=body_force)
            assert torch.equal(lat.f, c.f) and torch.equal(lat.nut, c.nut)
    for a, b in zip(*out):
        assert torch.equal(a, b)
