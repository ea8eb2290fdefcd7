"""The pressure boundary inside the step on rows that are no multiple of a
wavefront: boundary nodes fall on every lane, the first and the last among them
(taken by the launch before the step).  The same bytes as the separate kernels,
on both faces and in every storage form."""
import numpy as np
import pytest
import torch

import virtualfluids_amd as vfx
from tests import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("normal", [1, 2])
@pytest.mark.parametrize("nx", [5, 63, 64, 66, 70, 128, 130])
def test_every_lane_gives_the_separate_kernels_bytes(cuda, nx, normal, storage):
    print(f"[fused rows {nx} {normal} {storage}]", flush=True)
    dims = (nx, 9, 8)
    n = int(np.prod(dims))
    solid = np.zeros(dims[::-1], bool)
    solid[:, :, 0] = solid[:, :, -1] = True
    yz = nx * np.arange(9 * 8)
    nodes, inward = (yz + nx - 2, yz + nx - 3) if normal == 1 else (yz + 1, yz + 2)
    rho = 1e-3 * np.cos(np.arange(nodes.size))
    out = []
    for fuse in (False, True):
        lat = vfx.Lattice(dims, storage=storage, omega=1.9, solid=solid)
        lat.init_equilibrium(*cases.random_flow(dims, seed=nx))
        bc = vfx.BoundaryCondition(4, nodes, rho=rho, neighbors=inward, normal=normal)
        st = vfx.Stepper(lat, "k17", [bc], fuse=fuse)
        if fuse:  # the plan leaves entries with x mod 64 = 0 (63 for -x) to a kernel of their own
            assert (st.fused_plan().pre is None) == (normal == 1 and (nx - 2) % 64 == 0)
        st.step(5)
        st.step(2)
        out.append(lat.f.view(torch.uint8))
    assert torch.equal(*out)
    assert n == lat.n_nodes


def _call(lat, group, apply_pre):
    st, real = lat.struct(), lat._macro_dtype()
    g = group.struct(real)
    C = vfx._lib.C
    vfx.check(vfx.lib().vfx_k17_step_fused(C.byref(st), 1, None, 0, C.byref(g), None, apply_pre, None), "vfx_k17_step_fused")


@pytest.mark.parametrize("storage", ["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("fault", ["neighbour", "mask", "base"])
@pytest.mark.parametrize("normal", [1, 2])
def test_malformed_entries_select_nothing_on_every_lane(cuda, normal, fault, storage):
    """Entries whose neighbour is not the one beside them, or which the masks do
    not hold, leave the plain step's bytes wherever they lie in a wavefront."""
    print(f"[malformed {normal} {fault} {storage}]", flush=True)
    dims = (70, 9, 8)
    k = 70 * np.arange(72) + (68 if normal == 1 else 1)
    assert np.any(k % 64 == (0 if normal == 1 else 63))
    step = -1 if normal == 1 else 1
    out = []
    for malformed in (False, True):
        lat = vfx.Lattice(dims, storage=storage, omega=1.9)
        lat.init_equilibrium(*cases.random_flow(dims, seed=normal))
        if malformed:
            bc = vfx.BoundaryCondition(4, k, rho=1e-2 * np.ones(72), normal=normal,
                                       neighbors=k + (2 * step if fault == "neighbour" else step))
            g = vfx.FusedGroup(bc, lat.n_nodes)
            if fault == "mask":
                g.node_mask.zero_()
            if fault == "base":
                g.word_base += 1000
            _call(lat, g, 1)
        else:
            lat.collide_stream("k17", True)
        out.append(lat.f.view(torch.uint8))
    assert torch.equal(*out)


@pytest.mark.parametrize("storage", ["fp64", "fp32", "fp16"])
def test_without_the_launch_before_the_step(cuda, storage):
    """apply_pre -1 takes every entry but the ones whose neighbour lies in another
    wavefront; a group that has none is told so by itself."""
    print(f"[no edge launch {storage}]", flush=True)
    dims = (70, 9, 8)
    k = 70 * np.arange(72) + 68
    inside = k[k % 64 != 0]
    assert 0 < inside.size < k.size
    out = []
    for fused in (False, True):
        lat = vfx.Lattice(dims, storage=storage, omega=1.9)
        lat.init_equilibrium(*cases.random_flow(dims, seed=3))
        nodes = k if fused else inside
        bc = vfx.BoundaryCondition(4, nodes, rho=1e-2 * np.cos(nodes), neighbors=nodes - 1, normal=1)
        if fused:
            g = vfx.FusedGroup(bc, lat.n_nodes)
            assert g.edge and not vfx.FusedGroup(bc.subset(np.flatnonzero(k % 64)), lat.n_nodes).edge
            _call(lat, g, -1)
        else:
            lat.apply_bc(bc, True)
            lat.collide_stream("k17", True)
        out.append(lat.f.view(torch.uint8))
    assert torch.equal(*out)
