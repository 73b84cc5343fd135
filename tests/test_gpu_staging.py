"""Staged updates reach the store alike on every route: batches staged on the host threads
(with and without addresses named twice or already staged), single sends, updates applied
in the launch that predicts the others, and updates that change ids (which run before it).
An engine fed by single sends and flushed before each call is the reference: predicted
states, forces, nearest neighbours and lists are bit-identical to it, and the predicted
states equal the oracle's."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
import sapporo2_amd as sa
from _util import check_forces, load_engine, plummer_system, random_derivs

pytestmark = pytest.mark.gpu

# (updates, addresses repeated within the batch, addresses staged just before it, ids changed)
ROUNDS = [(1, 0, 0, 0), (63, 0, 0, 0), (64, 1, 0, 0), (65, 0, 2, 1), (255, 0, 0, 0), (256, 3, 0, 0), (257, 0, 0, 0),
          (1, 0, 0, 1), (256, 0, 9, 0), (0, 0, 0, 0), (2047, 0, 0, 0), (2048, 0, 0, 0),
          (2100, 0, 0, 3), (2500, 40, 0, 0), (2500, 0, 40, 0), (4099, 0, 0, 0), (6500, 30, 0, 0),
          (7000, 0, 0, 5), (6200, 0, 20, 0)]


@pytest.mark.parametrize("order", [sa.FOURTH, sa.SIXTH])
@pytest.mark.parametrize("prec", [sa.DOUBLESINGLE, sa.DOUBLE])
def test_update_routes_agree(order, prec):
    n = 7001
    m, x, v, ids, h2 = plummer_system(n, seed=71)
    ids = ids.copy()
    acc, jrk, snp, crk = random_derivs(n, 72, 0.3)
    if order < sa.SIXTH:
        snp = crk = None
    rng = np.random.Generator(np.random.PCG64(73))
    tj = -rng.uniform(0, 1.0 / 256, n)
    x, v = x.copy(), v.copy()
    opt = lambda a, q: None if a is None else a[q]  # noqa: E731
    with sa.Engine(order, prec) as a, sa.Engine(order, prec) as b:
        for e in (a, b):
            load_engine(e, m, x, v, ids, acc, jrk, snp, crk, tj=tj)
        for r, (nu, twice, before, newid) in enumerate(ROUNDS):
            print(f"staging order={order} prec={prec} round {r}: {nu} updates", flush=True)
            u = rng.choice(n, nu, replace=False)
            first = u[:before]                       # staged one by one just before the batch
            rep = rng.choice(u, twice, replace=False) if twice else u[:0]
            batch = np.concatenate([rep, u])         # the repeated ones come first: the last values win
            if newid:
                ids[u[-newid:]] = 100000 + 10 * r + np.arange(newid)
            xb = x.copy()
            x[u] += 1e-3 * rng.normal(size=(nu, 3))
            tj[u] = -rng.uniform(0, 1.0 / 512, nu)
            xs = np.concatenate([xb[rep] + 0.5, x[u]])
            for q in first:
                a.set_j_particle(q, ids[q], 0.0, 0.0, m[q], acc[q], jrk[q], v[q], xb[q] + 0.25, opt(snp, q),
                                 opt(crk, q))
            a.set_j_particles(batch, ids[batch], m[batch], xs, v[batch], acc[batch], jrk[batch], opt(snp, batch),
                              opt(crk, batch), tj=tj[batch])
            for q in u:
                b.set_j_particle(q, ids[q], tj[q], 0.0, m[q], acc[q], jrk[q], v[q], x[q], opt(snp, q), opt(crk, q))
            predict = r % 5 != 3
            ti = 1.0 / 512 * (1 + r % 3)
            for e in (a, b):
                e.set_time(ti) if predict else e.set_no_time()
            nj = n - 200 if r % 4 == 2 else n        # some updates lie beyond the predicted range
            b.force_prediction(nj)
            # small calls apply up to 256 updates in their force launch
            sel = np.sort(rng.choice(n, (150, 3, 32)[r % 3], replace=False))
            ai = acc[sel] if order >= sa.SIXTH else None
            res = []
            for e in (a, b):
                e.start_grav_calc(nj, ids[sel], x[sel], v[sel], 1e-4, h2[sel], ai=ai)
                g = e.get_grav_results(nj, len(sel))
                e.read_ngb_list()
                g["lists"] = [e.get_ngb_list(i)[:2] for i in range(len(sel))]
                res.append(g)
            for k in ("acc", "jrk", "pot", "nnb", "dsmin"):
                assert np.array_equal(res[0][k], res[1][k], equal_nan=True), (r, k)
            for (p, cp), (q, cq) in zip(res[0]["lists"], res[1]["lists"]):
                # a list past its 256 slots holds whichever ids came first
                assert cp == cq and (cp >= sa.NGB_CAP or np.array_equal(p, q)), r
            if predict and nj == n:                  # every address predicted to ti
                px, pv, pa = oracle.predict(order, ti, tj, x, v, acc, jrk, snp, crk)
                got = a.retrieve_predicted_j_particles(np.arange(n))
                assert np.array_equal(got["pos"], px) and np.array_equal(got["vel"], pv), r
                if order >= sa.SIXTH:
                    assert np.array_equal(got["acc"], pa), r


@pytest.mark.parametrize("prec", [sa.DOUBLESINGLE, sa.DOUBLE])
@pytest.mark.parametrize("n,upd,again", [(7001, 4096, 1000), (7001, 4096, 4095), (7001, 7001, 0), (4000, 4000, 0)])
def test_part_sent_early_and_all_updated(prec, n, upd, again):
    """Rows partly on the device when the launch that predicts reads them (4096 sends are
    copied ahead, sending one of them again takes back its row and those behind it), and
    every predicted particle an update, in one launch (4000) and in two (7001)."""
    m, x, v, ids, _ = plummer_system(n, seed=74)
    acc, jrk, _, _ = random_derivs(n, 75, 0.3)
    rng = np.random.Generator(np.random.PCG64(76))
    tj = -rng.uniform(0, 1.0 / 256, n)
    x = x.copy()
    with sa.Engine(sa.FOURTH, prec) as a:
        load_engine(a, m, x, v, ids, acc, jrk, tj=tj)
        a.force_prediction(n)
        print(f"staging prec={prec} n={n} updates={upd} again={again}", flush=True)
        u = np.sort(rng.choice(n, upd, replace=False))
        x[u] += 1e-3 * rng.normal(size=(upd, 3))
        for q in u:
            a.set_j_particle(q, ids[q], tj[q], 0.0, m[q], acc[q], jrk[q], v[q], x[q])
        if again:
            q = u[again]
            x[q] += 0.25
            a.set_j_particle(q, ids[q], tj[q], 0.0, m[q], acc[q], jrk[q], v[q], x[q])
        ti = 1.0 / 512
        a.set_time(ti)
        sel = np.sort(rng.choice(n, 100, replace=False))
        a.start_grav_calc(n, ids[sel], x[sel], v[sel], 1e-4)
        res = a.get_grav_results(n, len(sel))
        px, pv, _ = oracle.predict(sa.FOURTH, ti, tj, x, v, acc, jrk, None, None)
        got = a.retrieve_predicted_j_particles(np.arange(n))
        assert np.array_equal(got["pos"], px) and np.array_equal(got["vel"], pv)
        ref = oracle.force(sa.FOURTH, x[sel], v[sel], ids[sel], px, pv, m, ids, 1e-4)
        check_forces(res, ref, sa.FOURTH, 1e-6 if prec == sa.DOUBLESINGLE else 1e-12, label=f"n={n} updates={upd}")
