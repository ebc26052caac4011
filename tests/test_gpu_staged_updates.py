"""GPU: update tiles of supernodes of 128 columns and more, whose operands go through LDS,
against the oracle (remainders of tiles in every dimension)."""
import numpy as np
import pytest

import swcholesky_amd as S
from swcholesky_amd import api, problems as P
import oracle_py as O
from helpers import relF, setup

pytestmark = pytest.mark.gpu

# operator, panels per block of the right-looking steps (a block's last step has 64 columns
# for each)
CASES = {"dense_600": (lambda: P.dense_spd(600, seed=2), 8), "dense_641": (lambda: P.dense_spd(641, seed=2), 8),
         "dense_193": (lambda: P.dense_spd(193, seed=3), 2), "dense_330": (lambda: P.dense_spd(330, seed=3), 3),
         "lap3d_16": (lambda: P.laplacian3d_var(16, shift=1.0), 2), "vec3d_11": (lambda: P.vector3d_var(11), 8),
         "vec3d_9": (lambda: P.vector3d_var(9), 3)}


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("name", list(CASES))
def test_updates_of_many_columns_match_oracle(name, mode):
    make, rlb = CASES[name]
    prob = make()
    b, a2x, Lo, info = setup(prob)
    assert info == 0
    assert max(int(u["k"]) for u in api.build_fronts(b, rlb)["utiles"]) >= 128
    f = S.Factor(b, params=(rlb,))
    f.set_precision(mode)
    for rep in range(2):
        assert f.factor(prob.values) == 0
        L = f.L_values()
        if mode == 0:
            assert relF(L, Lo) < 1e-12
        else:
            L32, _ = O.factor(b, a2x, fp32_updates=True)
            assert relF(L, L32) < 10 * max(relF(L32, Lo), 1e-7)
            assert relF(L, Lo) < 10 * max(relF(L32, Lo), 1e-7)
