"""The threads that share host copies: started only by copies that have a part for them, as
many as the largest copy so far has parts, and arrays arrive whole whatever sizes follow each
other.  Host code only (hipstub: uploads fill the staging buffer that the next download of the
same array's length reads)."""

import pytest

import hipstub


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return hipstub.build(tmp_path_factory.mktemp("hipstub"))


SETUP = """
import os
PART, MOST = 256 << 10, min(8, len(os.sched_getaffinity(0)))
def threads():
    return len(os.listdir("/proc/self/task"))
def helpers(nbytes):
    return max(0, min(MOST, nbytes // PART) - 1)
lib()
"""


@pytest.mark.parametrize("nxp,nlev", [(3, 8), (17, 20), (20, 33), (40, 30)])
def test_threads_started(stub, nxp, nlev):
    out = hipstub.run(stub, SETUP + f"""
grid = abi.FortranGrid(M.build_mesh({nxp}), M.vertical_grid({nlev}))
""" + """
most = grid.mza * 4 * max(grid.mva, 2 * grid.mwa)       # the largest array: V fields, or volt
before = threads()
g = Context(grid, abi.make_params("f32", num_scalar=2, dtsm=300.0), device=0)
assert threads() - before == helpers(most), (threads() - before, helpers(most))
rng = np.random.default_rng(1)
for rep in range(200):
    a = rng.random((grid.mwa, grid.mza)).astype(np.float32)
    g.upload_scalar(1, a)
    assert np.array_equal(g.download_scalar(1).view(np.uint32), a.view(np.uint32)), rep
assert threads() - before == helpers(most)
g.close()
assert threads() == before
print("ok", helpers(most))
""")
    assert out.startswith("ok"), out
