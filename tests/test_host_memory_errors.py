"""Host memory that runs out inside a call ends in an error code, never in an abort: a
context is created, used and given back with the first, second, ... allocation of the call
failing, among them those of the threads that build its tables and copy its arrays.  Host
code only (hipstub)."""

import pytest

import hipstub


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return hipstub.build(tmp_path_factory.mktemp("hipstub"))


@pytest.mark.parametrize("prec,order,tracer", [("f32", 2, ""), ("f64", 3, ""), ("f32", 2, "patch")])
def test_create_without_host_memory(stub, prec, order, tracer):
    out = hipstub.run(stub, f"""
import os
os.environ["OLAMGPU_TRACER"] = {tracer!r}
grid = abi.FortranGrid(M.build_mesh(2), M.vertical_grid(4))
prm = abi.make_params({prec!r}, num_scalar=2, dtsm=300.0, order={order})
""" + """
Context(grid, prm, device=0).close()                # loads the library
n0 = stub.stub_news()
Context(grid, prm, device=0).close()
need = stub.stub_news() - n0
bad = 0
for k in range(1, need + 2):
    stub.stub_new_fail(k)
    try:
        Context(grid, prm, device=0).close()
    except OlamGpuError:
        bad += 1
    stub.stub_new_fail(0)
    Context(grid, prm, device=0).close()
assert bad > 0, need
print("ok", need, bad)
""")
    assert out.startswith("ok"), out
    print(out)
