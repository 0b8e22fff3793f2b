"""The Mindlin far field at other lengths: the proxy rings' matrices are built
for boxes of side 1, U(s x) = s (U(x) - x_3 log s) takes them to side s. A
mesh scaled by a power of two (the same octree), its single layer densities by
the inverse, has the same displacements and strains 1/a as large: the
reference's fixtures at their own size, 2^-20 and 2^13 times it.

Tolerance: the fixtures' own, 1e-10; the log term (log s up to 14) is 10 times
the others at most and costs one digit of 15."""
import numpy as np
import pytest

from conftest import load_golden, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,tag,iprec", [("hs_fault_p2", "", 2), ("hs_fault_p1", "", 1), ("hs_fault_low", "_p0", 0),
                                            ("hs_fault_low", "_m1", -1)])
@pytest.mark.parametrize("a", [2.0 ** -20, 1.0, 2.0 ** 13])
def test_scaled_mesh(gpu_lib, name, tag, iprec, a):
    g = load_golden(name)
    try:
        gpu_lib.half_parts(4)
        ier, _, pt, st = gpu_lib.elhfmm3dtriatargiter(
            iprec, float(g["lam"]), float(g["mu"]), a * g["triangle"], g["trinorm"], a * g["source"],
            g["sigma_sl"] / a, g["sigma_dl"], a * g["target"])
    finally:
        gpu_lib.half_parts(7)
    assert ier == 0
    assert rel(pt, g[f"mind{tag}_pt"]) < 1e-10 and rel(np.asarray(st) * a, g[f"mind{tag}_st"]) < 1e-10
