"""The calls a user of this library makes, as measurable cases.

A pass is one block step of a direct-summation integrator through the C-ABI of
libsapporo_amd.so, called as a compiled program calls it (arrays held by the caller, no
copies in between).  Three kinds of program:

* ``single``      one system: the previous active set is re-sent (set_j_particles), the block
                  time is set, the active particles' forces, nearest neighbours and, if wanted,
                  neighbour lists are computed and read back.  With ``predictors`` the active
                  particles are first picked up from the library's own predictor (the
                  6th-order flow).
* ``ensemble``    many independent clusters in one call.
* ``device``      the allocation-free call on device buffers (torch tensors, torch stream).

Outputs are everything the program reads.  Lists are read for ``read`` of the active
particles, evenly spread (an integrator asks for the lists of the particles whose
neighbourhood it has to rebuild, one call each).
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import sapporo2_amd as sa
from sapporo2_amd import ics

MAXLEN = sa.NGB_CAP
PIPES = sa.NPIPES
PREC = {"mixed": sa.DOUBLESINGLE, "fp64": sa.DOUBLE}
_dp = ctypes.POINTER(ctypes.c_double)
_ip = ctypes.POINTER(ctypes.c_int)


def _case(name, kind="single", order=4, prec="mixed", nj=131072, ni=1, resend=0, lists=True, read=0,
          model="plummer", predictors=False, clusters=0, lo=0, hi=0, frac=1.0, sizes_seed=0):
    c = dict(kind=kind, order=order, prec=prec, nj=nj, ni=ni, resend=resend, lists=lists, read=read, model=model,
             predictors=predictors, clusters=clusters, lo=lo, hi=hi, frac=frac, sizes_seed=sizes_seed)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest block step, the most frequent call of an individual-time-step run: one
        # particle is due, the one before it is re-sent
        _case("h4_step_1", ni=1, resend=1, read=1),
        # a binary's or small subsystem's step
        _case("h4_step_24", ni=24, resend=11, read=24),
        # an ordinary block, an odd count over a system that is no power of two
        _case("h4_step_333", nj=100003, ni=333, resend=150, read=16),
        # a large block with neighbour lists
        _case("h4_step_3000", ni=3000, resend=1500, read=64),
        # a full pipe of i-particles, the throughput call
        _case("h4_full_16384", ni=16384, resend=16384, read=256),
        # the same in all-FP64
        _case("h4_fp64_5000", prec="fp64", ni=5000, resend=2500, read=64),
        # a small star cluster with one shared step: every particle active, no lists
        _case("h4_shared_8192", nj=8192, ni=8192, resend=8192, lists=False),
        # 6th order, the predict / pick up / evaluate flow of its ABI, King model
        _case("h6_predictors_2500", order=6, nj=65536, ni=2500, resend=2500, lists=False, model="king",
              predictors=True),
        # 6th order in FP64 with lists
        _case("h6_fp64_777", order=6, prec="fp64", nj=30011, ni=777, resend=400, read=16),
        # many small clusters, each with a quarter of its stars due
        _case("ens_256", kind="ensemble", clusters=256, lo=256, hi=4096, frac=0.25, lists=False, sizes_seed=4),
        # data already on the GPU, nothing allocated
        _case("device_4096", kind="device", nj=65536, ni=4096, lists=False),
        # the largest: a million stars around a central mass
        _case("h4_million_16384", nj=(1 << 20) + 1, ni=16384, resend=8192, lists=False, model="plummer_bh"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["single"] * 6 + ["ensemble", "device"])
    order = rng.choice([4, 4, 4, 6])
    prec = rng.choice(["mixed", "mixed", "fp64"])
    if kind == "ensemble":
        n, lists = _logint(rng, 16, 256), rng.random() < 0.5
        return _case("", kind, order, prec, lists=lists, read=16 if lists else 0, clusters=n, lo=_logint(rng, 64, 256),
                     hi=_logint(rng, 512, 4096), frac=2.0 ** -rng.randint(0, 5), sizes_seed=rng.randrange(1 << 20))
    top = 262144 if prec == "mixed" and order == 4 else 131072
    nj = _logint(rng, 2048, top)
    ni = min(_logint(rng, 1, PIPES), nj)
    if kind == "device":
        return _case("", kind, order, prec, nj=nj, ni=ni, lists=False)
    lists = rng.random() < 0.6
    return _case("", kind, order, prec, nj=nj, ni=ni, resend=min(_logint(rng, 1, 2 * ni), nj), lists=lists,
                 read=min(ni, 16) if lists else 0, model=rng.choice(["plummer", "plummer", "king", "plummer_bh"]),
                 predictors=order == 6 and rng.random() < 0.5)


# --------------------------------------------------------------------------------------------
# Inputs (host arrays; the library's boundary takes host buffers).

def _sizes(case):
    return ics.ensemble_sizes(case["clusters"], case["lo"], case["hi"], seed=case["sizes_seed"])


def _eps2(case):
    return 1e-4 if case["kind"] == "ensemble" else 1e-6


def _model(name, n, seed):
    if name == "king":
        return ics.king(n, 6.0, seed=seed)
    if name == "plummer_bh":
        return ics.plummer_bh(n - 1, seed=seed)
    return ics.plummer(n, seed=seed)


def _taylor(x, v):
    """Derivatives of the motion in the Plummer mean field: the Taylor coefficients a program's
    corrector has stored for each particle."""
    r2 = (x * x).sum(1)[:, None] + ics.PLUMMER_SCALE ** 2
    w = r2 ** -1.5
    a = -w * x
    j = -w * v + 3.0 * ((x * v).sum(1)[:, None] / r2) * w * x
    return a, j, -w * a, -w * j


class Inputs:
    """Everything of one case that is made from the seed, before any library call."""

    def __init__(self, case, seed):
        rng = np.random.Generator(np.random.PCG64([seed, 17]))
        self.case = case
        h6 = case["order"] == 6
        if case["kind"] == "ensemble":
            self.sizes = _sizes(case)
            parts = [ics.plummer(int(n), seed=seed + 101 * c) for c, n in enumerate(self.sizes)]
            m, x, v = (np.concatenate([p[k] for p in parts]) for k in range(3))
            off, first = 0, []
            for n in self.sizes:  # each cluster starts at a multiple of 64 addresses
                first.append(off)
                off += -(-int(n) // 64) * 64
            self.addr = np.concatenate([f + np.arange(int(n)) for f, n in zip(first, self.sizes)]).astype(np.int32)
            start = np.concatenate([[0], np.cumsum(self.sizes)])
            sel = []
            for c, n in enumerate(self.sizes):
                k = max(1, int(n * case["frac"]))
                sel.append(start[c] + np.sort(rng.choice(int(n), k, replace=False)))
            self.cluster = np.concatenate([np.full(len(s), c) for c, s in enumerate(sel)]).astype(np.int32)
            self.act = np.concatenate(sel)
            self.start = start
            self.nj = len(m)
            self.eps2c = np.full(len(self.sizes), _eps2(case))
            h2 = np.concatenate([ics.neighbour_h2(p[1], 24.0) for p in parts])
            self.res = np.sort(rng.choice(self.nj, len(self.act), replace=False))  # re-sent
        else:
            self.nj = case["nj"]
            m, x, v = _model(case["model"], self.nj, seed)
            h2 = ics.neighbour_h2(x, 32.0)
            self.addr = np.arange(self.nj, dtype=np.int32)
            self.act = np.sort(rng.choice(self.nj, case["ni"], replace=False))
            self.res = np.sort(rng.choice(self.nj, case["resend"], replace=False))
        self.m, self.x, self.v = m, x, v
        self.a, self.j, self.s, self.c = _taylor(x, v)
        self.ids = (np.arange(self.nj) + 1).astype(np.int32)
        lev = ics.block_levels(self.nj, 20, seed=seed + 2)
        self.tj = -rng.uniform(0.0, 1.0, self.nj) * 2.0 ** -(3.0 + lev)
        # the program's own prediction of the particles to the block time t = 0
        dt = -self.tj[:, None]
        sn, cr = (self.s, self.c) if h6 else (0.0, 0.0)
        self.px = x + dt * (v + dt / 2 * (self.a + dt / 3 * (self.j + dt / 4 * (sn + dt / 5 * cr))))
        self.pv = v + dt * (self.a + dt / 2 * (self.j + dt / 3 * (sn + dt / 4 * cr)))
        self.pa = self.a + dt * (self.j + dt / 2 * (sn + dt / 3 * cr))
        self.h2 = h2


def _c(a, dtype=np.float64):
    return np.ascontiguousarray(a, dtype)


def _pd(a):
    return None if a is None else a.ctypes.data_as(_dp)


def _pi(a):
    return None if a is None else a.ctypes.data_as(_ip)


class State:
    """One program with its engine, its arrays and the pointers it passes."""

    stream = None  # the device program's one stream (its calls share the library's scratch region)

    def __init__(self, case, seed):
        d = self.data = Inputs(case, seed)
        self.case = case
        h6 = case["order"] == 6
        self.eng = sa.Engine(sa.SIXTH if h6 else sa.FOURTH, PREC[case["prec"]])
        self.L, self.h = sa.lib(), self.eng._h
        if case["kind"] == "ensemble":
            self.eng.set_clusters(d.sizes)
        self.eng.set_j_particles(d.addr, d.ids, d.m, d.x, d.v, d.a, d.j, d.s if h6 else None, d.c if h6 else None,
                                 tj=d.tj)
        self.eng.set_time(0.0)
        self.eng.force_prediction(d.nj)
        act, res = d.act, d.res
        ni = self.ni = len(act)
        self.nj = d.nj
        self.eps2 = _eps2(case)
        self.i_id = _c(d.ids[act], np.int32)
        self.i_x, self.i_v, self.i_a = _c(d.px[act]), _c(d.pv[act]), _c(d.pa[act])
        self.i_h2 = _c(d.h2[act]) if case["lists"] else None
        # a re-sent particle carries its state at the block time
        self.r_addr, self.r_id = _c(d.addr[res], np.int32), _c(d.ids[res], np.int32)
        self.r_m, self.r_t = _c(d.m[res]), np.zeros(len(res))
        self.r = [_c(q[res]) for q in (d.a, d.j, d.pv, d.px)] + ([_c(d.s[res]), _c(d.c[res])] if h6 else [])
        self.acc, self.jrk, self.snp = (np.zeros((ni, 3)) for _ in range(3))
        self.pot, self.dsmin, self.nnb = np.zeros(ni), np.zeros(ni), np.zeros(ni, np.int32)
        self.out = [self.acc, self.jrk] + ([self.snp] if h6 else []) + [self.pot, self.dsmin, self.nnb]
        # every pointer that the passes hand over
        self.a_resend = [len(res), _pi(self.r_addr), _pi(self.r_id), _pd(self.r_t), None, _pd(self.r_m),
                         *[_pd(q) for q in self.r], *([] if h6 else [None, None]), None]
        if case["kind"] == "ensemble":
            self.a_cl = [ni, _pi(d.cluster), _pi(self.i_id), _pd(self.i_x), _pd(self.i_v),
                         _pd(self.i_a) if h6 else None, _pd(d.eps2c), _pd(self.i_h2)]
        if case["predictors"]:
            self.p_addr, self.p_m = _c(d.addr[act], np.int32), np.zeros(ni)
            self.i_x, self.i_v, self.i_a = (np.zeros((ni, 3)) for _ in range(3))
            self.out += [self.p_m, self.i_x, self.i_v, self.i_a]
            self.a_pick = [ni, _pi(self.p_addr)] + [a.ctypes.data_as(ctypes.c_void_p)
                                                    for a in (self.p_m, self.i_x, self.i_v, self.i_a)]
        self.a_first = [d.nj, ni, _pi(self.i_id), _pd(self.i_x), _pd(self.i_v), _pd(self.i_a) if h6 else None,
                        self.eps2, _pd(self.i_h2)]
        self.a_last = [d.nj, ni, _pd(self.acc), _pd(self.jrk), _pd(self.snp) if h6 else None, None, _pd(self.pot),
                       _pi(self.nnb), _pd(self.dsmin), 1]
        self.read = min(case["read"], ni) if case["lists"] else 0
        if self.read:
            self.cnt, self.lst = np.zeros(self.read, np.int32), np.zeros((self.read, MAXLEN), np.int32)
            self.out += [self.cnt, self.lst]
            pipes = (np.arange(self.read) * ni) // self.read
            self.a_lists = [(int(p), MAXLEN, _pi(self.cnt[k:k + 1]), _pi(self.lst[k])) for k, p in enumerate(pipes)]
        if case["kind"] == "device":
            if State.stream is None:
                State.stream = torch.cuda.Stream()
            f = 13 if h6 else 10
            q = [self.i_x, self.i_v] + ([self.i_a] if h6 else [])
            self.d_id = torch.from_numpy(self.i_id).cuda()
            self.d_in = torch.from_numpy(np.concatenate([a.reshape(-1) for a in q])).cuda()
            self.d_out = torch.zeros((f, ni), dtype=torch.float64, device="cuda")
            # its rows: acc, pot, jerk, (snap,) smallest squared distance, its particle's id, 0
            cut = [0, 3, 4, 7] + ([10] if h6 else []) + [f - 2, f - 1, f]
            self.out = [self.d_out[b:e] for b, e in zip(cut, cut[1:]) if e > b]
            na = self.L.sapamd_grav_calc_noalloc
            na.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p,
                           ctypes.c_double, ctypes.c_void_p, ctypes.c_void_p]
            self.a_dev = [d.nj, ni, self.d_id.data_ptr(), self.d_in.data_ptr(), self.eps2, self.d_out.data_ptr(),
                          State.stream.cuda_stream]
            torch.cuda.synchronize()
        self.data = None


def prepare(case, seed):
    return State(case, seed)


def run(s):
    L, h = s.L, s.h
    kind = s.case["kind"]
    if kind == "device":
        rc = L.sapamd_set_time(h, 0.0)
        rc |= L.sapamd_grav_calc_noalloc(h, *s.a_dev)
        if rc:
            raise RuntimeError("grav_calc_noalloc failed")
        return s.out
    rc = L.sapamd_set_j_particles(h, *s.a_resend)
    rc |= L.sapamd_set_time(h, 0.0)
    if kind == "ensemble":
        rc |= L.sapamd_start_grav_calc_clusters(h, *s.a_cl)
    else:
        if s.case["predictors"]:
            rc |= L.sapamd_force_prediction(h, s.nj)
            rc |= L.sapamd_retrieve_predicted_j_particles(h, *s.a_pick)
        rc |= L.sapamd_start_grav_calc(h, *s.a_first)
    rc |= L.sapamd_get_grav_results(h, *s.a_last)
    if rc:
        raise RuntimeError("force call failed")
    if s.read:
        L.sapamd_read_ngb_list(h)
        get = L.sapamd_get_ngb_list
        for p, n, c, q in s.a_lists:
            get(h, p, n, c, q)
    return s.out


# --------------------------------------------------------------------------------------------

def work(case):
    h6 = case["order"] == 6
    if case["kind"] == "ensemble":
        n = _sizes(case)
        k = np.maximum(1, (n * case["frac"]).astype(np.int64))
        pairs, nj, ni = int((n * k).sum()), int(n.sum()), int(k.sum())
        resend = ni
    else:
        nj, ni, resend = case["nj"], case["ni"], case["resend"]
        pairs = ni * nj
    # j-particle: time, mass and the Taylor coefficients in FP64, the id; i-particle: position,
    # velocity (acceleration), radius and id in, the results out; a re-sent particle in and
    # into the store
    jb = (20 if h6 else 14) * 8 + 4
    ib = ((9 if h6 else 6) + (1 if case["lists"] else 0)) * 8 + 4 + ((10 if h6 else 7) + 1) * 8 + 4
    flops = (100.0 if h6 else 60.0) * pairs  # per interaction, the reference's convention
    return {"bytes": float(nj * jb + ni * ib + 2 * resend * jb), "flops": flops}


def tolerance(case):
    # About four times the whole-array errors measured against exact(): up to 9e-7 (mixed, snap;
    # its norm is carried by the closest pairs) and 1.3e-15 (FP64, snap).  Nearest neighbours,
    # counts and lists are whole numbers and do not differ.
    if case["prec"] == "fp64":
        return {"rel": 1e-14, "max": 1e-12}
    return {"rel": 4e-6, "max": 2e-4}


def _exact_forces(order, xi, vi, ai, idi, xj, vj, aj, mj, idj, eps2):
    """Direct sum in 64 bits over chunks of i-particles: acc, jerk, snap, pot and the smallest
    squared distance."""
    ni, nj = len(xi), len(xj)
    out = [torch.zeros((ni, 3), dtype=torch.float64, device=xj.device) for _ in range(3)]
    pot, ds = (torch.zeros(ni, dtype=torch.float64, device=xj.device) for _ in range(2))
    step = max(1, min(ni, (1 << 25) // nj))
    inf = float("inf")
    for b in range(0, ni, step):
        e = min(ni, b + step)
        d = [xj[None, :, k] - xi[b:e, None, k] for k in range(3)]
        u = [vj[None, :, k] - vi[b:e, None, k] for k in range(3)]
        r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
        same = idj[None, :] == idi[b:e, None]
        ds[b:e] = r2.masked_fill(same, inf).min(dim=1).values
        inv2 = 1.0 / (r2 + eps2).masked_fill(same, inf)
        inv = inv2.sqrt()
        w = mj[None, :] * inv
        pot[b:e] = -w.sum(dim=1)
        w = w * inv2
        al = (d[0] * u[0] + d[1] * u[1] + d[2] * u[2]) * inv2
        if order == 6:
            f = [aj[None, :, k] - ai[b:e, None, k] for k in range(3)]
            be = (u[0] * u[0] + u[1] * u[1] + u[2] * u[2] + d[0] * f[0] + d[1] * f[1] + d[2] * f[2]) * inv2 + al * al
        for k in range(3):
            out[0][b:e, k] = (w * d[k]).sum(dim=1)
            jk = w * (u[k] - 3.0 * al * d[k])
            out[1][b:e, k] = jk.sum(dim=1)
            if order == 6:
                out[2][b:e, k] = (w * (f[k] - 3.0 * be * d[k]) - 6.0 * al * jk).sum(dim=1)
    return out, pot, ds


def exact(case, seed):
    d = Inputs(case, seed)
    h6 = case["order"] == 6
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def t(a):
        return torch.from_numpy(np.ascontiguousarray(a)).to(dev)

    # the store at t = 0: predicted particles, the re-sent ones as sent (their acceleration is
    # the one they carry; the 4th-order forces do not use it)
    xj, vj, aj, mj, idj = t(d.px), t(d.pv), t(d.pa), t(d.m), t(d.ids)
    if h6 and case["kind"] != "device":
        aj[t(d.res)] = t(d.a[d.res])
    act = t(d.act)
    if case["predictors"]:
        xi, vi, ai = xj[act], vj[act], aj[act]
    else:
        xi, vi, ai = t(d.px)[act], t(d.pv)[act], t(d.pa)[act]
    idi = idj[act]
    if case["kind"] == "ensemble":
        got, at = [], 0
        for c in range(len(d.sizes)):
            b, e, k = int(d.start[c]), int(d.start[c + 1]), int((d.cluster == c).sum())
            i = slice(at, at + k)
            got.append(_exact_forces(case["order"], xi[i], vi[i], ai[i], idi[i], xj[b:e], vj[b:e], aj[b:e], mj[b:e],
                                     idj[b:e], float(d.eps2c[c])))
            at += k
        f = [torch.cat([g[0][k] for g in got]) for k in range(3)]
        pot, ds = torch.cat([g[1] for g in got]), torch.cat([g[2] for g in got])
    else:
        f, pot, ds = _exact_forces(case["order"], xi, vi, ai, idi, xj, vj, aj, mj, idj, _eps2(case))
    if case["kind"] == "device":
        out = [f[0].T, pot[None], f[1].T] + ([f[2].T] if h6 else []) + [ds[None], None, None]
        return [None if o is None else o.cpu() for o in out]
    out = [f[0], f[1]] + ([f[2]] if h6 else []) + [pot, ds, None]
    if case["predictors"]:
        out += [mj[act], xi, vi, ai]
    if case["lists"] and case["read"]:
        out += [None, None]
    return [None if o is None else o.cpu() for o in out]
