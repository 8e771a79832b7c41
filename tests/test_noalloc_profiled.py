"""olamgpu_mass_sums_noalloc takes no event, no device memory and no host memory of its own,
also while kernels are being timed, and olamgpu_mass_sums beside it is timed as before.  Host
code only (hipstub)."""

import pytest

import hipstub


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return hipstub.build(tmp_path_factory.mktemp("hipstub"))


@pytest.mark.parametrize("prec,ntr", [("f32", 0), ("mixed", 3), ("f64", 64)])
def test_noalloc_takes_nothing(stub, prec, ntr):
    out = hipstub.run(stub, f"""
grid = abi.FortranGrid(M.build_mesh(2), M.vertical_grid(4))
g = Context(grid, abi.make_params({prec!r}, num_scalar={ntr}), device=0)
""" + """
L, dev = lib(), np.zeros(65)
p = C.c_void_p(dev.ctypes.data)
for profiled in (False, True, True):
    g.set_profiling(profiled)
    if profiled:
        g.mass_sums()
        assert sorted(g.kernel_profile()) == ["k_mass_final", "k_mass_partial"]
    prof, at = g.kernel_profile(), stub.stub_launches()
    before = (stub.stub_mallocs(), stub.stub_events(), stub.stub_news())
    rc = L.olamgpu_mass_sums_noalloc(g.h, p)
    after = (stub.stub_mallocs(), stub.stub_events(), stub.stub_news())
    assert rc == 0 and after == before, (profiled, before, after)
    assert g.kernel_profile() == prof
    names = launches(at)
    assert len(names) == 2 and "k_mass_partial" in names[0] and "k_mass_final" in names[1], names
g2 = Context(grid, g.params, device=0)
g2.set_profiling(True)                              # nothing pooled from an earlier call
before = (stub.stub_mallocs(), stub.stub_events(), stub.stub_news())
assert L.olamgpu_mass_sums_noalloc(g2.h, p) == 0
assert (stub.stub_mallocs(), stub.stub_events(), stub.stub_news()) == before
print("ok")
""")
    assert out.startswith("ok")
