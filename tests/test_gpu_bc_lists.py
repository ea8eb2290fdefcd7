"""Boundary lists on both sides of the length at which their workgroups change
(65536 nodes): a long list leaves the bytes of its parts applied one by one."""
import numpy as np
import pytest
import torch

import virtualfluids_amd as vfx

pytestmark = pytest.mark.gpu

DIMS = (264, 260, 5)
PLANE = DIMS[0] * DIMS[1]


@pytest.mark.parametrize("storage", ["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("even", [True, False])
@pytest.mark.parametrize("kind", [1, 2, 3, 4, 5, 6])
def test_a_long_list_equals_its_parts(cuda, kind, even, storage):
    print(f"[list kind {kind} {even} {storage}]", flush=True)
    rng = np.random.default_rng(kind)
    nodes = PLANE + np.arange(PLANE)
    q = np.full((27, PLANE), -1.0)
    for d in range(1, 27):
        if vfx.CZ[d] < 0:
            q[d] = rng.uniform(0.0, 1.0, PLANE)
    kw = {}
    if kind in (2, 5):
        kw = dict(vx=rng.uniform(-0.05, 0.05, PLANE), vy=0.01, vz=0.0)
    if kind in (4, 6):
        kw = dict(rho=rng.uniform(-0.01, 0.01, PLANE), neighbors=nodes + PLANE, normal=6)
    bc = vfx.BoundaryCondition(kind, nodes, q, **kw)
    f = rng.uniform(-1e-2, 1e-2, 27 * 5 * PLANE)
    out = []
    for cuts in ([0, PLANE], [0, 64, 65536 - 1, PLANE], [0, 65536, PLANE]):
        lat = vfx.Lattice(DIMS, storage=storage, omega=1.7)
        lat.f.copy_(torch.from_numpy(f).to(lat.f.dtype))
        for a, b in zip(cuts, cuts[1:]):
            part = vfx.BoundaryCondition(kind, nodes[a:b], q[:, a:b], **{
                n: v[a:b] if isinstance(v, np.ndarray) else v for n, v in kw.items()})
            lat.apply_bc(part if b - a < PLANE else bc, even)
        out.append(lat.f.view(torch.uint8))
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
    assert not torch.equal(out[0].cpu(), torch.from_numpy(f).to(lat.f.dtype).view(torch.uint8))
