"""The choice between MFMA fragments and the plain matrix for unstructured
operators in ragged layouts (kernels._use_fragments) against both times, us,
measured on a card of 256 CUs."""

from types import SimpleNamespace

import pytest

from jaxfun_amd import kernels as K

# precision, M, K, P, Q, plain, fragments
MEASURED = [
    ("f64", 20, 10, 32, 2, 8.2, 7.9), ("f64", 40, 20, 81, 50, 12, 8), ("f64", 160, 80, 32768, 2, 92, 55),
    ("f64", 128, 192, 81, 50, 40, 17), ("f64", 128, 192, 524288, 2, 1770, 1628), ("f64", 192, 193, 65, 1000, 209, 180),
    ("f64", 224, 222, 81, 50, 47, 41), ("f64", 224, 222, 1310, 50, 243, 340), ("f64", 256, 254, 32, 2, 51, 35),
    ("f64", 256, 254, 65, 1000, 291, 380), ("f64", 30, 500, 8, 1000, 90, 51), ("f64", 30, 500, 1310, 50, 154, 456),
    ("f64", 100, 400, 32768, 2, 251, 351), ("f64", 400, 100, 32, 2, 25, 34), ("f64", 400, 100, 65, 1000, 228, 143),
    ("f64", 512, 40, 81, 50, 16, 24), ("f64", 512, 40, 655, 50, 67, 46), ("f64", 300, 298, 655, 50, 217, 341),
    ("f64", 512, 256, 1, 50, 51, 65), ("f64", 512, 510, 65, 1000, 1232, 3203), ("f32", 80, 40, 81, 50, 12, 8),
    ("f32", 224, 222, 32768, 2, 150, 117), ("f32", 100, 400, 81, 50, 59, 27), ("f32", 100, 400, 1310, 50, 122, 189),
    ("f32", 300, 298, 655, 50, 112, 161), ("f32", 400, 200, 81, 50, 35, 41), ("f32", 400, 200, 655, 50, 112, 90),
    ("f32", 512, 256, 1, 50, 38, 54), ("f32", 512, 510, 1310, 50, 483, 1042),
]


@pytest.mark.parametrize("prec,M,Kd,P,Q,plain,fragments", MEASURED)
def test_the_faster_one_is_chosen(prec, M, Kd, P, Q, plain, fragments):
    op = SimpleNamespace(M=M, K=Kd, parity=None, once=False)
    assert K._use_fragments(op, P, Q, prec) == (fragments < plain)
    assert K._use_fragments(SimpleNamespace(M=M, K=Kd, parity=K.evaluates_parity(), once=False), P, Q, prec)
