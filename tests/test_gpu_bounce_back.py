"""The bounce-back kernel (one thread per link or pair of links) on lists whose length sits at the
edges of a wavefront and a workgroup, with links chosen at random: every element
of the array against the formula, on the structured and the sparse layout, and
the boundary set's one-thread-per-node form against the kernel bit for bit."""
import numpy as np
import pytest
import torch

import virtualfluids_amd as vfx
from virtualfluids_amd import CX, CY, CZ, INV, W

pytestmark = pytest.mark.gpu

DIMS = (16, 16, 18)
N = int(np.prod(DIMS))


def _at(k, d, dims=DIMS):
    """The node direction d of node k lives on (one step along every axis with c_d < 0, periodic)."""
    nx, ny, nz = dims
    x, y, z = k % nx + (CX[d] < 0), k // nx % ny + (CY[d] < 0), k // (nx * ny) + (CZ[d] < 0)
    return x % nx + nx * (y % ny + ny * (z % nz))


def _case(n, seed):
    rng = np.random.default_rng(seed)
    # nodes with even coordinates: no link ends in another listed node, as no wall link of a grid does (the two
    # nodes' links would read and write one element)
    x, y, z = np.arange(N) % 16, np.arange(N) // 16 % 16, np.arange(N) // 256
    nodes = np.sort(rng.choice(np.flatnonzero((x % 2 == 0) & (y % 2 == 0) & (z % 2 == 0)), n, replace=False))
    q = np.where(rng.random((27, n)) < 0.4, rng.random((27, n)), -1.0)
    q[1, 0], q[2, 0], q[3, 0] = 0.0, 1.0, np.nan  # links at both ends of the range, and no link
    return nodes, q, rng.uniform(-0.05, 0.05, (3, n)), rng.uniform(-1e-2, 1e-2, 27 * N)


def _lattice(storage, sparse, f):
    if sparse:
        k = np.arange(N, dtype=np.uint32)
        nb = [_at(k, d).astype(np.uint32) for d in (2, 4, 6)]
        lat = vfx.Lattice(storage=storage, omega=1.7, neighbors=nb, fluid_nodes=k)
    else:
        lat = vfx.Lattice(DIMS, storage=storage, omega=1.7)
    lat.f.copy_(torch.from_numpy(f).to(lat.f.dtype))
    return lat


@pytest.mark.parametrize("even", [True, False])
@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 257])
def test_links_fp64(cuda, n, sparse, even):
    print(f"[bounce back {n} {sparse} {even}]", flush=True)
    nodes, q, u, f = _case(n, n)
    lat = _lattice("fp64", sparse, f)
    lat.apply_bc(vfx.BoundaryCondition(0, nodes, q, *u), even)
    ref = f.reshape(27, N).copy()
    for d in range(1, 27):
        on = (q[d] >= 0) & (q[d] <= 1)
        e = INV[d]
        at = _at(nodes[on], e)
        s = np.zeros(on.sum())
        first = True
        for c, v in zip((CX[d], CY[d], CZ[d]), u[:, on]):
            if c:
                s, first = (c * v if first else s + c * v), False
        ref[d if even else e, at] = f.reshape(27, N)[e if even else d, at] - 6.0 * W[d] * s
    got = lat.f.cpu().numpy().reshape(27, N)
    # 6 w rounded once here, 4/9, 1/9 and 1/36 in the kernel: one unit in the last place of a wall term <= 0.07
    assert np.abs(got - ref).max() <= 2e-17


@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_a_node_that_is_its_own_neighbour(cuda, axis, sparse):
    """A box one node thick with walls on both sides: a link and its opposite
    exchange their two populations, as the formula on the array before."""
    print(f"[bounce back axis {axis} {sparse}]", flush=True)
    dims = [8, 6, 16]
    dims[axis] = 1
    n = int(np.prod(dims))
    x = np.arange(n) % dims[0], np.arange(n) // dims[0] % dims[1], np.arange(n) // (dims[0] * dims[1])
    nodes = np.flatnonzero((x[0] % 2 == 0) & (x[1] % 2 == 0) & (x[2] % 2 == 0))
    f = np.random.default_rng(axis).uniform(-1e-2, 1e-2, 27 * n)
    if sparse:
        k = np.arange(n, dtype=np.uint32)
        lat = vfx.Lattice(storage="fp64", omega=1.7, neighbors=[_at(k, d, dims).astype(np.uint32) for d in (2, 4, 6)],
                          fluid_nodes=k)
    else:
        lat = vfx.Lattice(tuple(dims), storage="fp64", omega=1.7)
    lat.f.copy_(torch.from_numpy(f))
    lat.apply_bc(vfx.BoundaryCondition(0, nodes, np.full((27, nodes.size), 0.5)), True)
    ref = f.reshape(27, n).copy()
    for d in range(1, 27):
        at = _at(nodes, INV[d], dims)
        ref[d, at] = f.reshape(27, n)[INV[d], at]
    assert np.array_equal(lat.f.cpu().numpy().reshape(27, n), ref)


@pytest.mark.parametrize("storage", ["fp64", "fp32", "fp16"])
@pytest.mark.parametrize("even", [True, False])
def test_pairs_give_the_single_links_bytes(cuda, even, storage):
    """A sparse list none of whose nodes is its own neighbour runs a thread per
    link, any other a thread per pair: the same bytes."""
    print(f"[bounce back single {even} {storage}]", flush=True)
    nodes, q, u, f = _case(257, 5)
    bc = vfx.BoundaryCondition(0, nodes, q, *u)
    out = []
    for single in (1, 0):
        lat = _lattice(storage, True, f)
        s, b = lat.struct(), lat._bc_struct(bc)
        assert b.single_links == 1
        b.single_links = single
        C = vfx._lib.C
        vfx.check(vfx.lib().vfx_bc_apply(C.byref(s), C.byref(b), int(even), None), "vfx_bc_apply")
        out.append(lat.f.view(torch.uint8))
    assert torch.equal(*out)


@pytest.mark.parametrize("storage", ["fp64", "fp32", "fp16"])
def test_set_gives_the_kernels_bits(cuda, storage):
    print(f"[bounce back set {storage}]", flush=True)
    nodes, q, u, f = _case(130, 3)
    a, b = _lattice(storage, False, f), _lattice(storage, False, f)
    bc = vfx.BoundaryCondition(0, nodes, q, *u)
    a.apply_bc(bc, True)
    vfx.BCSet([(b, bc)]).apply([True])
    assert torch.equal(a.f.view(torch.uint8), b.f.view(torch.uint8))
