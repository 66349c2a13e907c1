"""FP64 operator products against recorded ones.  The rounding of the bases is
part of the product: directions that the pivoted MGS leaves small are their
rounding errors' size, so that bases of the same span made with sums in another
order move a product by 1e-14 to 1e-13 of its norm, 1e-11 at tighter SVD
tolerances.  The bases keep their order of sums; what may differ is the order of
the apply's own FP64 sums, a few hundred terms of 1.1e-16 each: 4e-15 of the
root mean square entry."""
import json
import os
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
sys.path.insert(0, GOLDEN)

import make_fp64_products as rec  # noqa: E402

REF = json.load(open(os.path.join(GOLDEN, "fp64_products.json")))


@pytest.mark.parametrize("name", list(rec.CASES))
def test_products(name):
    norm, y = rec.product(name)
    ref = np.array([float.fromhex(v) for v in REF[name]["entries"]])
    assert abs(norm - float.fromhex(REF[name]["norm"])) <= 4e-15 * norm
    assert np.linalg.norm(y - ref) <= 4e-15 * np.linalg.norm(ref)
