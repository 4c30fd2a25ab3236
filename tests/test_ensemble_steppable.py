"""Which instances take whole steps: the array form equals the rule, side by side."""

import itertools

import numpy as np

from finitevolumegpu_amd.Ensemble import steppable
from finitevolumegpu_amd.Simulator import BoundaryCondition

T = BoundaryCondition.Type


def test_steppable_of_every_edge_combination():
    kinds = (T.Dirichlet, T.Periodic, T.Reflective, T.Outflow)
    table = [(nx, ny, edges) for nx in (7, 8, 300) for ny in (2, 8, 9) for edges in itertools.product(kinds, repeat=4)]
    codes = [int(BoundaryCondition(dict(zip(("north", "south", "east", "west"), e))).asCodedInt()) for _, _, e in table]
    got = steppable(*(np.array(c, dtype=np.int32) for c in ([t[0] for t in table], [t[1] for t in table], codes)))
    for (nx, ny, (n, s, e, w)), code, g in zip(table, codes, got):
        want = (nx >= 8 and ny >= 8 and T.Dirichlet not in (n, s, e, w)
                and (n == T.Periodic) == (s == T.Periodic) and (e == T.Periodic) == (w == T.Periodic))
        assert bool(g) is want and bool(steppable(nx, ny, code)) is want
    assert steppable(*(np.zeros(0, dtype=np.int32),) * 3).all()
