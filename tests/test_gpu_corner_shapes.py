"""Corner terms of sheared blocks one, two and three cells thick along each axis: thin blocks take the walks
around their corners, the others the direct loads; both against the oracle, as in
test_gpu_assembly.test_nonortho_assembly_matches_oracle (same operators and flags). FP64 only: the
relative bound of that test holds no room for cancellation, and on four cells the divergence is the
difference of fluxes ~100 times its size, 4e-6 of it in FP32."""
from __future__ import annotations

import numpy as np
import pytest

import cases
from oracle import oracle as O
from test_gpu_assembly import test_nonortho_assembly_matches_oracle as check_operators

pytestmark = pytest.mark.gpu


def _sheared(specs):
    v = specs[0].vertices.copy()
    v[0] += 0.3 * v[1]
    if v.shape[0] == 3:
        v[1] += 0.2 * v[2]
        v[0] += 0.1 * v[2]
    specs[0].vertices = v
    return specs


@pytest.mark.parametrize("flags", [O.NO_DEFAULT_MODE, O.NO_DEFAULT_MODE | O.NO_DIRECT_RHS])
@pytest.mark.parametrize("sizes", [(1, 4), (4, 1), (2, 3), (3, 2), (65, 3), (2, 1, 3), (3, 2, 2), (1, 3, 4), (66, 2, 3)],
                         ids=lambda s: "x".join(map(str, s)))
def test_thin_blocks(sizes, flags, monkeypatch):
    make = cases.channel2d if len(sizes) == 2 else cases.duct3d
    monkeypatch.setitem(cases.CASES, "thin", lambda: _sheared(make(*sizes)))
    check_operators("thin", flags, np.float64)
