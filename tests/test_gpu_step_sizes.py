"""The structured step on boxes whose rows, slabs and node count do not fit its
tiles or wavefronts, against the CPU checker: FP64 reproduces it bit for bit.
The sizes sit at the edges of the flat node mapping (one node in a direction,
rows of one node more or less than a wavefront, a last tile of one node)."""
import numpy as np
import pytest

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
