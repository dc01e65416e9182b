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


WAYS = {"direct": 1, "mixed": 0, "walked": 2}


@pytest.mark.parametrize("case,chosen,ways", [
    ("channel", "direct", ("direct", "mixed", "walked")), ("duct", "direct", ("direct", "mixed", "walked")),
    ("wide pair", "mixed", ("mixed", "walked")), ("junction", "walked", ("mixed", "walked")),
    ("slab", "walked", ("mixed", "walked")),
])
def test_every_way_around_the_corners(case, chosen, ways, monkeypatch):
    """The kernels with direct loads, with walks and with both, on each domain they may be used for, against the
    oracle; and the one that the domain chooses. The wide pair and the junction have wavefronts (64
    consecutive cells) with cells at a connection and others without."""
    import torch

    from phipict_amd.domain import Domain

    make = {"channel": lambda: cases.channel2d(70, 5), "duct": lambda: cases.duct3d(66, 3, 4),
            "wide pair": lambda: cases.split_channel2d(400, 4, 200)[1], "junction": lambda: cases.tjunction3d(16),
            "slab": lambda: _sheared(cases.duct3d(1, 9, 30))}[case]
    dom = cases.build_domain(cases.skew(make(), 0.25, seed=7), 0.02, 0.01, torch.float64)
    assert dom._corner_ways() == WAYS[chosen]
    monkeypatch.setitem(cases.CASES, "ways", make)
    for way in ways:
        monkeypatch.setattr(Domain, "_corner_ways", lambda self, w=WAYS[way]: w)
        check_operators("ways", O.NO_DEFAULT_MODE | O.NO_DIRECT_RHS, np.float64)
