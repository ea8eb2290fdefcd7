"""Which calls a Stepper makes: a lattice or boundary that replaces a launch is
stepped through its own, every step, and a precursor's reader may change the
lattice between steps.  No GPU: the library is a recorder."""
import numpy as np
import pytest

import virtualfluids_amd as vfx
from tests.test_geometry import small_channel
from tests.test_oracle_refinement import small_cube_case
from virtualfluids_amd import _lib, geometry, lattice

DIMS = (6, 5, 4)
LAUNCHES = ("collide_stream", "apply_bc", "turbulent_viscosity_amd")


class Library:
    """Stands in for libvfx: notes each call's name, parity and the lattice's omega."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(lat, *args):
            self.calls.append((name, lat._obj.omega))
            return 0
        return call


@pytest.fixture
def library(monkeypatch):
    lib = Library()
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    monkeypatch.setattr(lattice, "_stream", lambda stream: stream)
    return lib


def _bounce():
    return vfx.BoundaryCondition(0, [7, 8], np.full((27, 2), 0.5), device="cpu")


def _outlet():
    return vfx.BoundaryCondition(4, [10], rho=[0.0], neighbors=[9], normal=1, device="cpu")


def _expected(model):
    step = ["collide_stream", "apply_bc"] + (["turbulent_viscosity_amd"] if model == "amd" else []) + ["apply_bc"]
    return step * 3


@pytest.mark.parametrize("model", ["none", "amd"])
@pytest.mark.parametrize("where", ["subclass", "instance", "class"])
def test_a_replaced_launch_is_called(library, monkeypatch, where, model):
    seen = []

    def noting(name):
        original = getattr(vfx.Lattice, name)

        def method(*args, **kw):
            seen.append(name)
            return original(*args, **kw)
        return method

    new = {n: noting(n) for n in LAUNCHES}
    cls = type("Noting", (vfx.Lattice,), new) if where == "subclass" else vfx.Lattice
    if where == "class":
        for n in LAUNCHES:
            monkeypatch.setattr(vfx.Lattice, n, new[n])
    lat = cls(DIMS, storage="fp32", omega=1.5, device="cpu", turbulence=model, sgs_constant=0.1)
    if where == "instance":
        for n in LAUNCHES:
            setattr(lat, n, new[n].__get__(lat))
    vfx.Stepper(lat, "k17", [_bounce(), _outlet()]).step(3)
    assert seen == _expected(model)
    assert len(library.calls) == len(seen)


def test_a_boundary_with_its_own_tables_makes_them_every_step(library):
    class Pulsating(vfx.BoundaryCondition):
        made = 0

        def struct(self, real):
            self.made += 1
            return super().struct(real)

    bc = Pulsating(0, [7, 8], np.full((27, 2), 0.5), device="cpu")
    vfx.Stepper(vfx.Lattice(DIMS, storage="fp32", omega=1.5, device="cpu"), "k17", [bc]).step(4)
    assert bc.made == 4


def test_a_reader_may_change_the_lattice(library):
    lat = vfx.Lattice(DIMS, storage="fp32", omega=1.5, device="cpu")

    def reader(time):
        lat.omega += 0.01
        return np.zeros((3, 2))

    planes = vfx.PrecursorPlanes(np.zeros((4, 1), int), np.full((4, 1), 0.25), 2, 3, reader=reader, device="cpu",
                                 real=lat._macro_dtype())
    lat.omega = 1.5
    bc = vfx.BoundaryCondition(12, [7], np.full((27, 1), 0.5), precursor=planes, device="cpu")
    vfx.Stepper(lat, "k17", [_bounce(), bc]).step(4)
    omegas = [o for name, o in library.calls if name == "vfx_collide_stream"]
    # planes are read from the first time step on: each step's collision sees what the reads before it left
    assert omegas == pytest.approx([1.5, 1.51, 1.52, 1.53])


@pytest.mark.parametrize("own,nodes,single", [(None, [3, 7], 1), (0, [3, 7], 1), (9, [3, 7], 1), (7, [3, 7], 0),
                                              (5, [3, 7], 0)])
def test_sparse_lists_say_when_no_node_is_its_own_neighbour(library, own, nodes, single):
    """own: a node that is its own neighbour along y; a list whose node numbers
    lie on one side of all such nodes holds none of them."""
    n = 12
    k = np.arange(n, dtype=np.uint32)
    y = (k + 3) % n
    if own is not None:
        y[own] = own
    lat = vfx.Lattice(storage="fp32", omega=1.5, neighbors=[(k + 1) % n, y, (k + 5) % n], fluid_nodes=k, device="cpu",
                      regular_groups=False)
    bc = vfx.BoundaryCondition(0, nodes, np.full((27, 2), 0.5), device="cpu")
    assert lat._bc_struct(bc).single_links == single
    assert vfx.Lattice((3, 4, 1), storage="fp32", omega=1.5, device="cpu")._bc_struct(bc).single_links == 0


def test_plain_lattices_make_one_view(library, monkeypatch):
    lat = vfx.Lattice(DIMS, storage="fp32", omega=1.5, device="cpu")
    made = []
    b = _bounce()
    b.tables(lat._macro_dtype())
    original = vfx.Lattice.struct

    def struct(self):
        made.append(1)
        return original(self)

    monkeypatch.setattr(vfx.Lattice, "struct", struct)
    monkeypatch.setitem(lattice._LATTICE_LAUNCHES, "struct", struct)
    vfx.Stepper(lat, "k17", [b]).step(5)
    assert len(made) == 1
    assert [n for n, _ in library.calls] == ["vfx_collide_stream", "vfx_bc_apply"] * 5


@pytest.mark.parametrize("fuse_post", [True, False])
def test_fused_steps_run_other_boundaries_whole(library, fuse_post):
    """One launch per boundary that is not inside the step, in the listed order,
    also where only some of its entries could be a group of the step's call."""
    ch = small_channel()
    solid = ch.solid.copy()
    wall = next(t for t in ch.bcs if t.kind == 1)
    k, d = int(wall.nodes[0]), int(np.flatnonzero(wall.q27[:, 0] >= 0)[0])
    nx, ny, nz = ch.dims
    x, y, z = (k % nx + vfx.CX[d]) % nx, (k // nx % ny + vfx.CY[d]) % ny, (k // (nx * ny) + vfx.CZ[d]) % nz
    solid[x + nx * (y + ny * z)] = False  # this entry's link ends in a fluid node
    seen = []

    class Noting(vfx.Lattice):
        def k17_step_fused(self, even, post=(), pre=None, apply_pre=False, any_mask=None, stream=None):
            seen.append((list(post), pre is not None, any_mask))

        def apply_bc(self, bc, even=True, stream=None):
            seen.append(bc)

    bcs = geometry.boundary_conditions(ch.bcs, device="cpu")
    st = vfx.Stepper(Noting(ch.dims, storage="fp32", omega=1.5, solid=solid, device="cpu"), "k17", bcs, fuse=True,
                     fuse_post=fuse_post)
    assert vfx.FusedPlan.build(st.lattice, bcs).residual_post
    st.step(2)
    post = [b for b in bcs if not b.pre_collision]
    assert len(post) == 2
    outlet = seen.pop()
    assert outlet.kind == 4 and outlet.n == next(b for b in bcs if b.pre_collision).n
    assert seen == [([], True, None)] + post + [([], True, None)] + post


def test_plans_make_their_tables(monkeypatch):
    """A step may be captured right after fused_plan() or a RefinedStepper with
    fuse_outlet: the boundaries a plan splits off have their tables by then."""
    ch = small_channel()
    lat = vfx.Lattice(ch.dims, storage="fp32", omega=1.5, solid=ch.solid, device="cpu")
    st = vfx.Stepper(lat, "k17", geometry.boundary_conditions(ch.bcs, device="cpu"), fuse=True)
    st.fused_plan()
    monkeypatch.setattr(vfx.FusedPlan, "build", None)
    plan = st._plan(False)
    assert lat._macro_dtype() in plan.pre.bc._dev
    monkeypatch.undo()
    case = small_cube_case()
    r = vfx.RefinedStepper(case.nest, case.omega, storage="fp32", device="cpu", coarse_solid=case.coarse_solid,
                           fine_solid=case.fine_solid, fuse_outlet=True,
                           coarse_bcs=geometry.boundary_conditions(case.coarse_bcs, device="cpu"),
                           fine_bcs=geometry.boundary_conditions(case.fine_bcs, device="cpu"))
    parts = [r._plan_c.pre.bc] + r._plan_c.residual_pre + r._plan_c.residual_post
    assert all(r.coarse._macro_dtype() in b._dev for b in parts)
