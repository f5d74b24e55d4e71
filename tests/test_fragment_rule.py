"""Choices of kernels by size against the times of both sides, us, measured on a
card of 256 CUs: MFMA fragments or the plain matrix for unstructured operators in
ragged layouts (kernels._use_fragments), slab kernel or one launch per axis
(kernels.slab_pays)."""

from types import SimpleNamespace

import pytest
import torch

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


# M0, K0, M1, K1, slabs, slab kernel, per axis
SLABS = [(64, 62, 64, 62, 1, 10, 15), (66, 64, 66, 64, 16, 13, 16), (80, 78, 80, 78, 1, 15.3, 16.2),
         (64, 62, 128, 126, 100, 15.4, 18.1), (126, 128, 62, 64, 1, 15.5, 16.5), (20, 18, 128, 126, 1, 9.4, 16.8),
         (94, 96, 31, 33, 100, 11, 17), (2, 3, 126, 128, 16, 9.9, 17.7), (96, 94, 96, 94, 1, 17.8, 16.3),
         (96, 94, 96, 94, 128, 20, 23), (128, 126, 128, 126, 16, 27, 17), (128, 126, 128, 126, 200, 31, 43)]


@pytest.mark.parametrize("M0,K0,M1,K1,slabs,fused,separate", SLABS)
def test_the_faster_slab_pass_is_chosen(monkeypatch, M0, K0, M1, K1, slabs, fused, separate):
    monkeypatch.setattr(K, "num_cus", lambda: 256)
    ops = [K.AxisOperator(torch.zeros(s, dtype=torch.float64), K.evaluates_parity()) for s in ((M0, K0), (M1, K1))]
    assert K.slab_pays(*ops, slabs) == (fused < separate)
    assert K.slab_pays(ops[0], K.AxisOperator(ops[1].A64), slabs) is None
