"""Launch shapes of the force call at their edges against the oracle: active counts around
the i-group and finalize boundaries, j counts around the pair loop's sub-blocks and tiles,
splits with nothing in them, records taken ahead or not, and i-particles with most of the
system inside their radius (exact counts past a full list).  Forces within the precision's
tolerance, nearest neighbours, counts and lists bit-exact."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import sapporo2_amd as sa
from _util import check_forces, check_nn_lists, load_engine, plummer_system

pytestmark = pytest.mark.gpu
TOL = {sa.DOUBLESINGLE: 1e-6, sa.DOUBLE: 1e-12}


def _check(eng, order, prec, sys_, sel, nj, lists, label):
    m, x, v, ids, h2 = sys_
    print(label, flush=True)
    ai = np.zeros((len(sel), 3)) if order >= sa.SIXTH else None
    eng.start_grav_calc(nj, ids[sel], x[sel], v[sel], 1e-4, h2[sel] if lists else None, ai=ai)
    res = eng.get_grav_results(nj, len(sel))
    aj = np.zeros((nj, 3)) if order >= sa.SIXTH else None
    ref = oracle.force(order, x[sel], v[sel], ids[sel], x[:nj], v[:nj], m[:nj], ids[:nj], 1e-4, h2=h2[sel], ai=ai,
                       aj=aj)
    check_forces(res, ref, order, TOL[prec] * (10 if order >= sa.SIXTH else 1), label=label)
    if lists:
        check_nn_lists(eng, res, prec == sa.DOUBLE, x[sel], ids[sel], x[:nj], ids[:nj], h2[sel], label=label)


@pytest.mark.parametrize("order", [sa.FOURTH, sa.SIXTH])
@pytest.mark.parametrize("prec", [sa.DOUBLESINGLE, sa.DOUBLE])
def test_counts_at_shape_edges(order, prec):
    n = 9000
    m, x, v, ids, h2 = plummer_system(n, seed=91)
    h2 = h2.copy()
    h2[::7] = 4.0                                   # most of the system
    rng = np.random.Generator(np.random.PCG64(92))
    sys_ = (m, x, v, ids, h2)
    with sa.Engine(order, prec) as eng:
        load_engine(eng, m, x, v, ids, np.zeros((n, 3)), np.zeros((n, 3)),
                    *([np.zeros((n, 3))] * 2 if order >= sa.SIXTH else [None, None]))
        eng.set_time(0.0)
        for ni, nj in [(1, 1), (1, 255), (2, 256), (3, 257), (5, 4097), (8, 1000), (17, 9000), (31, 2047), (32, 8991), (63, 5000), (33, 1), (33, 15), (40, 16), (64, 17), (65, 63), (65, 80), (128, 1000), (129, 4097), (512, 8991),
                       (513, 9000), (1025, 2047), (4097, 3000)]:
            sel = np.sort(rng.choice(n, ni, replace=False))
            _check(eng, order, prec, sys_, sel, nj, ni % 2 == 1, f"shapes order={order} prec={prec} ni={ni} nj={nj}")


@pytest.mark.parametrize("prec", [sa.DOUBLESINGLE, sa.DOUBLE])
@pytest.mark.parametrize("S", [1, 3, 16, 33, 200])
def test_split_counts(prec, S):
    """Forced j-splits, among them more than there are sub-blocks (empty splits)."""
    n = 2500
    sys_ = plummer_system(n, seed=93)
    m, x, v, ids, h2 = sys_
    with sa.Engine(sa.FOURTH, prec) as eng:
        load_engine(eng, m, x, v, ids)
        eng.set_time(0.0)
        eng.set_force_override(64, S)
        sel = np.arange(0, n, 19)
        _check(eng, sa.FOURTH, prec, sys_, sel, n, True, f"splits prec={prec} S={S}")


@pytest.mark.parametrize("order", [sa.FOURTH, sa.SIXTH])
def test_mixed_without_records_ahead(order):
    """More waves than take their records ahead in mixed precision (4096): the kernel of
    large calls, at counts that leave remainders of i-groups, splits and tiles."""
    n = 9000
    m, x, v, ids, h2 = plummer_system(n, seed=94)
    h2 = h2.copy()
    h2[::7] = 4.0                                   # most of the system
    rng = np.random.Generator(np.random.PCG64(95))
    z = np.zeros((n, 3))
    with sa.Engine(order, sa.DOUBLESINGLE) as eng:
        load_engine(eng, m, x, v, ids, z, z, *([z, z] if order >= sa.SIXTH else [None, None]))
        eng.set_time(0.0)
        for ni, nj, lists in [(4097, 8991, True), (4097, 8991, False), (8191, 8999, True), (6001, 8977, False)]:
            sel = np.sort(rng.choice(n, ni, replace=False))
            _check(eng, order, sa.DOUBLESINGLE, (m, x, v, ids, h2), sel, nj, lists, f"full chip order={order} ni={ni} nj={nj}")
            P, S, _ = eng.last_config()
            assert P == 64 and (ni + 63) // 64 * S > 4096
