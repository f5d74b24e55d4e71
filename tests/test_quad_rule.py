"""The choice between the fused quadratic term and separate launches
(IMEXRungeKutta._quad_pays) against both times, measured on a card of 256 CUs."""

from types import SimpleNamespace

import pytest

from jaxfun_amd import kernels as K
from jaxfun_amd.integrators.imex_rk import IMEXRungeKutta

# precision, mesh points, problems, us fused, us separate
MEASURED = [
    ("f64", (64, 64), 1, 19, 69), ("f64", (128, 128), 1, 66, 67), ("f64", (144, 144), 90, 99, 110),
    ("f64", (192, 192), 32, 157, 110), ("f64", (192, 192), 90, 158, 176), ("f64", (192, 192), 300, 328, 392),
    ("f64", (129, 192), 32, 129, 97), ("f64", (176, 176), 200, 168, 261), ("mixed", (129, 129), 90, 100, 163),
    ("mixed", (33, 192), 128, 60, 80), ("mixed", (64, 192), 160, 69, 77), ("mixed", (64, 192), 400, 102, 122),
    ("mixed", (96, 192), 128, 77, 85), ("mixed", (96, 192), 300, 147, 131), ("mixed", (96, 192), 512, 151, 167),
    ("mixed", (128, 192), 128, 113, 99), ("mixed", (128, 192), 200, 114, 132), ("mixed", (128, 192), 300, 219, 154),
    ("mixed", (129, 192), 90, 131, 104), ("mixed", (129, 192), 256, 132, 154), ("mixed", (129, 192), 400, 257, 218),
    ("mixed", (144, 192), 160, 132, 117), ("mixed", (160, 192), 128, 144, 122), ("mixed", (160, 192), 300, 282, 192),
    ("mixed", (176, 192), 768, 475, 438), ("mixed", (192, 192), 160, 163, 148), ("mixed", (192, 192), 256, 163, 181),
    ("mixed", (192, 192), 300, 317, 222), ("mixed", (192, 128), 160, 100, 182), ("mixed", (192, 64), 128, 47, 96),
    ("mixed", (96, 256), 200, 120, 206), ("mixed", (64, 256), 768, 260, 380),
]


@pytest.mark.parametrize("precision,Np,batch,fused,separate", MEASURED)
def test_the_faster_one_is_chosen(monkeypatch, precision, Np, batch, fused, separate):
    monkeypatch.setattr(K, "num_cus", lambda: 256)
    it = SimpleNamespace(Np=Np, precision="f64" if precision == "f64" else "bf16x6",
                         testspace=[SimpleNamespace(dim=round(q / 1.5) - 2) for q in Np])
    assert IMEXRungeKutta._quad_pays(it, batch) == (fused < separate)
