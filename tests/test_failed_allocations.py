"""A device allocation that fails leaves a call that can be repeated: it fails again while
the memory is missing and launches nothing that would use it, allocates what is missing once
memory is there, and does not spoil the calls after it.  Host code only: the HIP runtime is a
stand-in (hipstub) whose allocations the test makes fail one after the other."""

import pytest

import hipstub


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return hipstub.build(tmp_path_factory.mktemp("hipstub"))


SETUP = """
grid = abi.FortranGrid(M.build_mesh(3), M.vertical_grid(8))
def context(**kw):
    g = Context(grid, abi.make_params("f32", num_scalar=2, dtsm=300.0, **kw), device=0)
    g.scalar_transport_rk()
    return g
w = np.zeros((grid.mwa, grid.mza), np.float32)
i = np.zeros(grid.mwa, np.int32)
"""

CALLS = {
    "adjoint": ("context(scal_order={order})", "lambda: g.scalar_transport_rk_adj()"),
    "upload_scalar_adj": ("context(scal_order={order})", "lambda: g.upload_scalar_adj(1, w)"),
    "set_nudging": ("context()", "lambda: g.set_nudging(wmanud=w)"),
    "set_turbulence": ("context()", "lambda: g.set_turbulence(w, w, i, i, w[:, 0].copy())"),
}


@pytest.mark.parametrize("call,order", [("adjoint", 2), ("adjoint", 3), ("adjoint", 1), ("upload_scalar_adj", 2),
                                        ("set_nudging", 2), ("set_turbulence", 2)])
def test_call_after_failed_allocation(stub, call, order):
    make, f = CALLS[call]
    make = make.format(order=order).replace("scal_order", "order")
    out = hipstub.run(stub, SETUP + f"""
g = {make}
n0 = stub.stub_mallocs()
({f})()
need = stub.stub_mallocs() - n0
g.close()
assert need > 1, need
for k in range(need):
    g = {make}
    f = {f}
    stub.stub_malloc_ok(k)
    assert "out of memory" in (fails(f) or ""), k
    at = stub.stub_launches()
    for again in range(2):
        assert "out of memory" in (fails(f) or ""), (k, "no error the next time", launches(at))
    assert not any(x in n for n in launches(at) for x in ("k_tr_vr", "ring2_adj", "k_tr_adj", "horiz_k")), launches(at)
    stub.stub_malloc_ok(-1)
    at = stub.stub_mallocs()
    g.scalar_transport_rk()                 # a call without allocations, after the failure
    f()
    assert stub.stub_mallocs() - at == need - k, (k, stub.stub_mallocs() - at, need)
    f()
    assert stub.stub_mallocs() - at == need - k
    g.close()
print("ok", need)
""")
    assert out.startswith("ok")


def test_create_after_failed_allocation(stub):
    out = hipstub.run(stub, SETUP + """
n0 = stub.stub_mallocs()
context().close()
need = stub.stub_mallocs() - n0
for k in range(need):
    stub.stub_malloc_ok(k)
    assert "out of memory" in (fails(context) or ""), k
    stub.stub_malloc_ok(-1)
    context().close()
print("ok", need)
""")
    assert out.startswith("ok")
