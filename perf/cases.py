"""Workloads of the track-building path, for timing and for comparing two builds of the library.

Each case is one call sequence that a program linked against mkfit_amd makes on data already on the GPU:
batched and per-slot track fits, the single propagation / update operations, the hit sort plus a track
finder over one event or a batch of events, one layer step of a caller's own layer loop, the backward fit
and the gradient of the fit.  Inputs come from the toy Monte Carlo; where a case needs more tracks or
events than are quick to generate, they are repeated turned about the beam line by random angles, which
the barrel and the disks leave as likely as the originals.

`exact` evaluates the same propagation, material and update formulas in 64 bits with torch.
"""
import math

import numpy as np
import torch

import mkfit_amd as mk

DEV = "cuda:0"
BFIELD = 3.8
BASE_TRACKS = 12000      # tracks generated on the host per batch; larger batches turn them about the beam
BASE_EVENTS = 3          # finding events generated on the host per batch

# FP32 operations (oracle/flopcount.cc): one barrel and one endcap step with material and chi2, the gradient's
# forward + reverse step, and per seed and layer the finders' work on 2 noise hits / cm^2.
FLOP_BARREL, FLOP_ENDCAP = 1394, 581
FLOP_SEED_LAYER = {"ce": 4.7e4, "std": 5.5e4, "bh": 1.6e3}


def listed():
    return [
        # A handful of blocks of tracks fitted on their own, as a per-event trigger path does: latency.
        {"name": "fit_small", "kind": "fit", "form": "batched", "n": 1003, "geometry": 1, "ordered": False,
         "fallback": False, "pca": False},
        # The uneven production batch: barrel and endcap, 8-30 hits, missing layers, FP64 fallback, packed by length.
        {"name": "fit_uneven_large", "kind": "fit", "form": "batched", "n": 1_000_000, "geometry": 3, "ordered": True,
         "fallback": True, "pca": False},
        # The per-layer form on an even barrel batch, with the step to the closest approach.
        {"name": "fit_plain_barrel", "kind": "fit", "form": "plain", "n": 200_003, "geometry": 2, "ordered": False,
         "fallback": False, "pca": True},
        # The MPlex free functions called one by one by a caller's own loop.
        {"name": "mplex_ops", "kind": "ops", "n": 500_009},
        # One small event, best hit per layer.
        {"name": "find_bh_small", "kind": "find", "finder": "bh", "n": 500, "events": 1, "noise": 1.0, "disks": False,
         "max_cands": 1, "mask": False, "material": False, "prop_to_hit": False},
        # One ordinary event through the clone engine.
        {"name": "find_ce_event", "kind": "find", "finder": "ce", "n": 10_000, "events": 1, "noise": 2.0,
         "disks": False, "max_cands": 6, "mask": False, "material": False, "prop_to_hit": True},
        # One event through standard finding in a later iteration: hits taken earlier are masked.
        {"name": "find_std_event", "kind": "find", "finder": "std", "n": 5_003, "events": 1, "noise": 2.0,
         "disks": False, "max_cands": 4, "mask": True, "material": True, "prop_to_hit": True},
        # Offline batches: 50 events in one load and one launch.
        {"name": "find_ce_batch", "kind": "find", "finder": "ce", "n": 10_000, "events": 50, "noise": 2.0,
         "disks": False, "max_cands": 6, "mask": False, "material": False, "prop_to_hit": True},
        {"name": "find_bh_batch", "kind": "find", "finder": "bh", "n": 10_000, "events": 50, "noise": 2.0,
         "disks": False, "max_cands": 1, "mask": False, "material": False, "prop_to_hit": False},
        # One layer of a caller's own layer loop: propagate, select, candidates, best hit.
        {"name": "finder_layer", "kind": "layer", "n": 30_011, "noise": 2.0, "layer": 6},
        # Backward fit of every found candidate of a batch of events.
        {"name": "backward_fit", "kind": "bkfit", "n": 160_000, "events": 16, "group": 16, "pca": True},
        # Alignment: gradient of the fit's chi2 with respect to material and offsets.
        {"name": "adjoint", "kind": "adjoint", "n": 100_000, "fp64": False, "every": 5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fit", "fit", "ops", "find", "find", "find", "find", "layer", "bkfit", "adjoint"])
    if kind == "fit":
        form = rng.choice(["batched", "batched", "plain"])
        geometry = rng.choice([1, 2, 3])
        return {"kind": "fit", "form": form, "n": _log_int(rng, 200, 700_000 if form == "batched" else 200_000),
                "geometry": geometry, "ordered": rng.random() < 0.5, "fallback": rng.random() < 0.5,
                "pca": rng.random() < 0.3}
    if kind == "ops":
        return {"kind": "ops", "n": _log_int(rng, 100, 500_000)}
    if kind == "find":
        finder = rng.choice(["ce", "std", "bh"])
        disks = rng.random() < 0.25
        return {"kind": "find", "finder": finder, "n": _log_int(rng, 300, 4_000 if disks else 15_000),
                "events": _log_int(rng, 1, 12), "noise": round(rng.uniform(0.2, 2.0), 2), "disks": disks,
                "max_cands": 1 if finder == "bh" else rng.randint(2, 8), "mask": rng.random() < 0.3,
                "material": not disks and rng.random() < 0.3,
                "prop_to_hit": finder != "bh" or rng.random() < 0.4}
    if kind == "layer":
        return {"kind": "layer", "n": _log_int(rng, 300, 30_000), "noise": round(rng.uniform(0.5, 2.0), 2),
                "layer": rng.randint(3, 14)}
    if kind == "bkfit":
        events = rng.randint(1, 12)
        return {"kind": "bkfit", "n": _log_int(rng, 500, 10_000) * events, "events": events,
                "group": rng.choice([1, 8, 16, 64]), "pca": rng.random() < 0.7}
    return {"kind": "adjoint", "n": _log_int(rng, 500, 90_000), "fp64": rng.random() < 0.3,
            "every": rng.choice([3, 5, 8])}


# ---------------------------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------------------------

def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _rng(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _turn_xy(x, y, c, s):
    return c * x - s * y, s * x + c * y


def _turn_cov(xx, yx, yy, zx, zy, c, s):
    """A symmetric (xx, yx, yy, zx, zy, .) block turned about z."""
    return (c * c * xx - 2 * c * s * yx + s * s * yy, c * s * (xx - yy) + (c * c - s * s) * yx,
            s * s * xx + 2 * c * s * yx + c * c * yy, c * zx - s * zy, s * zx + c * zy)


def _wrap(phi):
    return torch.where(phi >= math.pi, phi - 2 * math.pi, torch.where(phi < -math.pi, phi + 2 * math.pi, phi))


def _spread(ev, n, seed, min_hits=0):
    """The generated tracks `ev` (host arrays, fit layout) of at least min_hits hits as n tracks on the GPU: beyond
    the generated ones, random tracks of the batch turned by random angles."""
    if min_hits:
        ev = {k: v[..., ev["n_hits"] >= min_hits] for k, v in ev.items()}
    m = ev["seed_par"].shape[1]
    keep = [k for k in ("seed_par", "seed_err", "chg", "hit_pos", "hit_err", "n_hits", "hit_flags", "hit_layer",
                        "truth_par") if k in ev]
    t = {k: _gpu(ev[k]) for k in keep}
    if n <= m:
        return {k: v[..., :n].contiguous() for k, v in t.items()}
    g = _rng(seed)
    idx = torch.randint(0, m, (n,), generator=g, device=DEV)
    ang = (torch.rand(n, generator=g, device=DEV) * 2 - 1) * math.pi
    c, s = torch.cos(ang), torch.sin(ang)
    t = {k: v[..., idx] for k, v in t.items()}
    for k in ("seed_par", "truth_par"):
        if k in t:
            p = t[k]
            x, y = _turn_xy(p[..., 0, :], p[..., 1, :], c, s)
            p[..., 0, :], p[..., 1, :], p[..., 4, :] = x, y, _wrap(p[..., 4, :] + ang)
    hp, he = t["hit_pos"], t["hit_err"]
    hp[:, 0], hp[:, 1] = _turn_xy(hp[:, 0], hp[:, 1], c, s)
    he[:, 0], he[:, 1], he[:, 2], he[:, 3], he[:, 4] = _turn_cov(he[:, 0], he[:, 1], he[:, 2], he[:, 3], he[:, 4], c, s)
    return t                                     # the generator's seed covariance is diagonal, equal in x and y


def _fit_tracks(case, seed):
    geo = mk.geometry(case["geometry"])
    if case["geometry"] == 3:
        params = mk.default_toy_params(seed=seed, bfield=BFIELD, eta_max=2.5, hits_min=8, hits_max=30, missing_frac=0.05)
        slots = 30
    else:
        params = mk.default_toy_params(seed=seed, bfield=BFIELD)
        slots = geo.n_barrel
    ev = _spread(mk.generate(geo, params, min(case["n"], BASE_TRACKS), slots), case["n"], seed)
    if case["ordered"]:                          # mkfit_amd.fit_order's key: hit count, then the endcap slots
        s = torch.arange(slots, device=DEV)[:, None]
        ec = ((ev["hit_flags"] & mk.HIT_ENDCAP) != 0) & (s < ev["n_hits"][None])
        key = (ev["n_hits"].long() << 40) | (ec.long() << s).sum(0)
        perm = torch.argsort(key, stable=True)
        ev = {k: v[..., perm].contiguous() for k, v in ev.items()}
    return geo, ev


def _no_material(ev):
    return (ev["n_hits"] < ev["hit_pos"].shape[0]).int()     # any per-track choice: the tracks that stop early


def _find_event(geo, case, seed, n):
    p = mk.default_toy_params(seed=seed, simulate_material=int(case.get("material", False)))
    if case.get("disks"):
        p = mk.default_toy_params(seed=seed, simulate_material=0, eta_max=2.5, pt_min=1.0)
    # About a third of the tracks reach three disks; n of the seeds are kept.
    ev = mk.generate_find_event(geo, p, n * 7 // 2 + 40 if case.get("disks") else n + n // 50 + 8,
                                noise_per_cm2=case["noise"])
    if ev["n_seeds"] < n:
        raise RuntimeError("the toy event holds %d seeds, not %d" % (ev["n_seeds"], n))
    for k in ("seed_par", "seed_err", "seed_chg", "seed_hits"):
        ev[k] = np.ascontiguousarray(ev[k][..., :n])
    return dict(ev, n_seeds=n)


def _find_inputs(case, seed):
    """Hits and seeds of the case's events: host offsets and batch dict, device hits [total, 9]."""
    geo = mk.geometry(4 if case.get("disks") else 1)
    descs = mk.disk_layer_descs(geo) if case.get("disks") else mk.barrel_layer_descs(geo)
    L, E = len(descs), case.get("events", 1)
    lo, hi = (case["n"], case["n"]) if E == 1 else (case["n"] // 2, case["n"] + case["n"] // 2)
    rng = np.random.default_rng(seed)
    sizes = np.linspace(lo, hi, min(E, BASE_EVENTS)).astype(int)
    base = [_find_event(geo, case, seed * 31 + e, int(m)) for e, m in enumerate(sizes)]
    dev = [_gpu(b["hits_flat"]) for b in base]
    evs, hits = [], []
    for e in range(E):
        b, h = base[e % len(base)], dev[e % len(base)]
        if e >= len(base):
            a = float(rng.uniform(-math.pi, math.pi))
            c, s = math.cos(a), math.sin(a)
            h = h.clone()
            h[:, 0], h[:, 1] = _turn_xy(h[:, 0].clone(), h[:, 1].clone(), c, s)
            h[:, 3], h[:, 4], h[:, 5], h[:, 6], h[:, 7] = _turn_cov(*(h[:, k].clone() for k in range(3, 8)), c, s)
            sp = b["seed_par"].copy()
            sp[0], sp[1] = _turn_xy(b["seed_par"][0], b["seed_par"][1], np.float32(c), np.float32(s))
            phi = b["seed_par"][4] + np.float32(a)
            sp[4] = np.where(phi >= math.pi, phi - 2 * math.pi, np.where(phi < -math.pi, phi + 2 * math.pi, phi))
            b = dict(b, seed_par=sp)
        evs.append(b)
        hits.append(h)
    cnt = np.concatenate([np.diff(b["hit_offset"]) for b in evs])
    cat = {"hit_offset": np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32),
           "n_seeds": sum(b["n_seeds"] for b in evs)}
    for k in ("seed_par", "seed_err", "seed_hits", "seed_chg"):
        cat[k] = np.concatenate([b[k] for b in evs], axis=-1)
    cat["layer_base"] = np.concatenate([np.full(b["n_seeds"], e * L, np.int32) for e, b in enumerate(evs)])
    return geo, descs, cat, hits[0] if E == 1 else torch.cat(hits)


def _context(geo, material):
    rl, xi = mk.material_grid(geo) if material else (None, None)
    return mk.Context(bfield=BFIELD, rl_grid=rl, xi_grid=xi, device=0)


def _disk_tracks(n, seed):
    geo = mk.geometry(4)
    params = mk.default_toy_params(seed=seed, bfield=BFIELD, eta_max=2.5, pt_min=1.0)
    return _spread(mk.generate(geo, params, min(n, BASE_TRACKS) + 64, geo.n_disk), n, seed, min_hits=2)


def _barrel_tracks(n, seed):
    geo = mk.geometry(2)
    params = mk.default_toy_params(seed=seed, bfield=BFIELD)
    return geo, _spread(mk.generate(geo, params, min(n, BASE_TRACKS) + 64, geo.n_barrel), n, seed, min_hits=2)


def _bk_inputs(case, seed):
    """Found candidates as the finders leave them: the tracks of a 17-layer barrel, each with its hit on every
    layer or a hole, their state on the last layer, and events of hits that hold those hits among noise."""
    geo = mk.geometry(1)
    L, E, n = geo.n_barrel, case["events"], case["n"]
    params = mk.default_toy_params(seed=seed, bfield=BFIELD, pt_min=0.8, hits_min=8, hits_max=L)   # no loopers
    ev = _spread(mk.generate(geo, params, min(n, BASE_TRACKS) + 600, L, truth=True), n, seed, min_hits=5)
    g = _rng(seed + 1)
    nh = ev["n_hits"].long()
    event = torch.arange(n, device=DEV) * E // n                  # contiguous runs of candidates per event
    hot = torch.full((L, n), -9, dtype=torch.int32, device=DEV)
    hits, offset = [], [0]
    slot = torch.arange(L, device=DEV)[:, None]
    valid = slot < nh[None]
    holes = torch.rand((L, n), generator=g, device=DEV) < 0.06
    per_slot = torch.cat([ev["hit_pos"], ev["hit_err"]], 1)       # [slot][9][n]
    for e in range(E):
        tr = (event == e).nonzero()[:, 0]
        for l in range(L):
            on = valid[:, tr] & (ev["hit_layer"][:, tr] == l)     # the slot holding the track's layer-l hit
            s = on.int().argmax(0)
            here = on.any(0)
            own = tr[here]
            h = per_slot[s[here], :, own]
            hot[l, own] = torch.arange(len(own), device=DEV, dtype=torch.int32)
            r, zm = geo.barrel_r[l], geo.barrel_zmax[l]
            m = int(round(2 * math.pi * r * 2 * zm * 0.5))
            ph = torch.rand(m, generator=g, device=DEV) * (2 * math.pi)
            z = (torch.rand(m, generator=g, device=DEV) * 2 - 1) * zm
            zero = torch.zeros_like(z)
            c, sn = torch.cos(ph), torch.sin(ph)
            noise = torch.stack([r * c, r * sn, z, 1e-4 * sn * sn, -1e-4 * sn * c, 1e-4 * c * c, zero, zero, zero + 1e-2], 1)
            hits += [h, noise]
            offset.append(offset[-1] + len(own) + m)
    keep = (hot >= 0).long().cumsum(0).sub((hot >= 0).long()) < 3  # a seed's hits are never holes
    hot = torch.where((hot >= 0) & holes & ~keep, torch.full_like(hot, -1), hot)
    last = (nh.clamp(min=1) - 1)
    truth = ev["truth_par"][last, :, torch.arange(n, device=DEV)].T.contiguous()
    sig = torch.tensor([0.004, 0.004, 0.04, 0.0, 1e-3, 1e-3], device=DEV)[:, None].repeat(1, n)
    sig[3] = 0.02 * truth[3].abs()
    par = truth + sig * torch.randn((6, n), generator=g, device=DEV)
    par[3], par[4] = par[3].abs(), _wrap(par[4])
    err = torch.zeros((21, n), device=DEV)
    for i in range(6):
        err[i * (i + 1) // 2 + i] = sig[i] ** 2
    base = (event * L).int()
    return geo, np.array(offset, np.int32), torch.cat(hits).contiguous(), \
        {"par": par, "err": err, "chg": ev["chg"], "hot_idx": hot}, base


def _adjoint_inputs(case, seed):
    from mkfit_amd.alignment import make_event
    ev, _, theta = make_event(min(case["n"], BASE_TRACKS), seed=seed)
    return _spread(ev, case["n"], seed), theta.astype(np.float32)


class _Events:
    """What a program keeps for finding: context, layers, hits and the batch."""


def prepare(case, seed):
    kind = case["kind"]
    if kind == "fit":
        geo, ev = _fit_tracks(case, seed)
        ctx = _context(geo, True)
        flags = mk.FIT_CHI2 | mk.FIT_CHARGE_FLIP * case["pca"] | mk.FIT_FP64_FALLBACK * case["fallback"] | \
            mk.FIT_PROP_TO_PCA * case["pca"]
        out = [torch.zeros_like(ev[k]) for k in ("seed_par", "seed_err", "chg")]
        batch = mk.FitBatch(*out, torch.zeros(case["n"], dtype=torch.float32, device=DEV), ev["hit_pos"], ev["hit_err"],
                            ev["n_hits"], ev["hit_flags"], pflags=mk.PF_APPLY_MATERIAL, fit_flags=flags,
                            seed=(ev["seed_par"], ev["seed_err"], ev["chg"]), pca_pflags=0)
        return ctx, case["form"], batch
    if kind == "ops":
        geo, ev = _barrel_tracks(case["n"], seed)
        disk = _disk_tracks(case["n"], seed)
        n = case["n"]
        like = lambda *shape: torch.zeros(*shape, n, dtype=torch.float32, device=DEV)
        barrel = dict(err=ev["seed_err"], par=ev["seed_par"], chg=ev["chg"], mp=ev["hit_pos"][1].contiguous(),
                      me=ev["hit_err"][1].contiguous(), no_mat=_no_material(ev))
        barrel["r"] = torch.hypot(barrel["mp"][0], barrel["mp"][1])
        endcap = dict(err=disk["seed_err"], par=disk["seed_par"], chg=disk["chg"], mp=disk["hit_pos"][1].contiguous(),
                      me=disk["hit_err"][1].contiguous())
        fail = torch.zeros(n, dtype=torch.int32, device=DEV)
        out = [(like(21), like(6), like(21), like(6), like()) for _ in range(2)]
        return _context(geo, True), barrel, endcap, fail, out
    if kind == "find":
        geo, descs, cat, hits = _find_inputs(case, seed)
        s = _Events()
        s.ctx = _context(geo, case["material"])
        s.eoh = mk.EventOfHits(s.ctx, descs * case["events"])
        s.offset, s.hits, s.finder = cat["hit_offset"], hits, case["finder"]
        pf = mk.PF_APPLY_MATERIAL if case["material"] else 0
        base = cat["layer_base"] if case["events"] > 1 else None
        if case["finder"] == "bh":
            s.batch = mk.FindBatch(cat, len(descs), 3, device=DEV, chi2_cut=15.0, pflags=pf,
                                   prop_to_hit=case["prop_to_hit"], layer_base=base)
        else:
            s.batch = mk.CEBatch(cat, len(descs), 3, device=DEV, chi2_cut=30.0, max_cands=case["max_cands"], pflags=pf,
                                 prop_to_hit=case["prop_to_hit"], layer_base=base)
        s.mask = (torch.rand(hits.shape[0], generator=_rng(seed), device=DEV) < 0.05).to(torch.uint8) \
            if case["mask"] else None
        return s
    if kind == "layer":
        geo, descs, cat, hits = _find_inputs(dict(case, events=1), seed)
        s = _Events()
        s.ctx = _context(geo, False)
        s.eoh = mk.EventOfHits(s.ctx, descs)
        s.eoh.load(cat["hit_offset"], hits)
        n = cat["n_seeds"]
        s.layer = case["layer"]
        s.par, s.err, s.chg = _gpu(cat["seed_par"]), _gpu(cat["seed_err"]), _gpu(cat["seed_chg"])
        # A track that has hits on the layers before: the seed's covariance shrunk to the update's.
        s.err = s.err * torch.linspace(0.05, 0.2, n, device=DEV)
        s.r = torch.full((n,), descs[s.layer]["propagate_to"], dtype=torch.float32, device=DEV)
        s.found = torch.full((n,), s.layer, dtype=torch.int32, device=DEV)
        s.lanes = mk.FinderLanes(torch.zeros_like(s.par), torch.zeros_like(s.err), s.chg, n_found=s.found)
        i32 = lambda *shape: torch.zeros(*shape, dtype=torch.int32, device=DEV)
        s.xsize, s.xarr, s.wsr, s.code, s.n_entries = i32(n), i32(mk.HIT_IDX_MAX, n), i32(n), i32(n), i32(n)
        s.entries = torch.zeros(n * mk.CE_ENTRIES_PER_LANE * mk.IDX_CHI2_DTYPE.itemsize, dtype=torch.uint8, device=DEV)
        return s
    if kind == "bkfit":
        geo, offset, hits, cand, base = _bk_inputs(case, seed)
        s = _Events()
        s.ctx = _context(geo, False)
        s.eoh = mk.EventOfHits(s.ctx, mk.barrel_layer_descs(geo) * case["events"])
        s.eoh.load(offset, hits)
        s.batch = mk.BkFitBatch(cand, device=DEV, group=case["group"], pflags=mk.PF_USE_PARAM_B_FIELD,
                                pca_pflags=mk.PF_USE_PARAM_B_FIELD, include_pca=case["pca"], layer_base=base)
        return s
    ev, theta = _adjoint_inputs(case, seed)
    ctx = mk.Context(bfield=BFIELD, device=0)
    host = {k: np.zeros((1,) + tuple(1 for _ in ev[k].shape[1:]), np.float32) for k in ("hit_pos", "hit_err")}
    data = mk.AlignmentData(ctx, dict(host, seed_par=np.zeros((6, 1), np.float32), seed_err=np.zeros((21, 1), np.float32),
                                      chg=np.zeros(1, np.int32), n_hits=np.zeros(1, np.int32)),
                            DEV, checkpoint_every=case["every"], fp64=case["fp64"])
    # the device arrays of the batch, already there
    data.n, data.n_layers = case["n"], ev["hit_pos"].shape[0]
    data.seed_par, data.seed_err, data.seed_chg = ev["seed_par"], ev["seed_err"], ev["chg"]
    data.hit_pos, data.hit_err, data.n_hits = ev["hit_pos"], ev["hit_err"], ev["n_hits"]
    data.chi2 = torch.zeros(data.n, dtype=torch.float32, device=DEV)
    data.grad = torch.zeros((data.n_layers, 3), dtype=torch.float32, device=DEV)
    return data, _gpu(theta)


def run(state):
    if isinstance(state, _Events):
        s = state
        if hasattr(s, "finder"):
            s.eoh.load(s.offset, s.hits)
            if s.mask is not None:
                s.eoh.set_hit_mask(s.mask)
            if s.finder == "bh":
                s.batch.reset()
                s.ctx.find_tracks_best_hit(s.eoh, s.batch)
                return [getattr(s.batch, k) for k in ("par", "err", "chg", "chi2", "hot_idx", "n_found")]
            (s.ctx.find_tracks_clone_engine if s.finder == "ce" else s.ctx.find_tracks_standard)(s.eoh, s.batch)
            return [getattr(s.batch, k) for k in ("n_cands", "par", "err", "chg", "chi2", "score", "n_found", "hot_idx")]
        if hasattr(s, "lanes"):
            ln = s.lanes
            ln.chg.copy_(s.chg)
            ln.n_found.copy_(s.found)
            for k in ("chi2", "n_inside_minus_one", "n_tail_minus_one"):
                getattr(ln, k).zero_()
            s.ctx.propagate_helix_to_r(s.err, s.par, s.chg, s.r, ln.prop_err, ln.prop_par)
            s.eoh.select_hit_indices(s.layer, ln.prop_par, ln.prop_err, s.xsize, s.xarr, s.wsr)
            s.ctx.find_candidates_clone_engine(s.eoh, s.layer, ln, s.xsize, s.xarr, s.wsr, s.n_entries, s.entries)
            s.ctx.add_best_hit(s.eoh, s.layer, ln, s.xsize, s.xarr, s.wsr, s.code)
            rec = s.entries.view(torch.int32).view(-1, 12)           # IDX_CHI2_DTYPE: words 7..10 are floats
            return [s.xsize, s.xarr, s.wsr, s.code, s.n_entries, rec[:, :7], rec[:, 7:11].view(torch.float32), rec[:, 11],
                    *(getattr(ln, k) for k in ln.KEYS)]
        s.ctx.backward_fit(s.eoh, s.batch)
        return [getattr(s.batch, k) for k in ("par", "err", "chg", "chi2", "score")]
    if isinstance(state[0], mk.AlignmentData):
        data, theta = state
        return list(data.run(theta))
    if len(state) == 3:
        ctx, form, b = state
        (ctx.fit_batched if form == "batched" else ctx.fit_plain)(b)
        return [b.par, b.err, b.chg, b.chi2]
    ctx, barrel, endcap, fail, ((e0, p0, ue0, up0, c0), (e1, p1, ue1, up1, c1)) = state
    both = mk.KFO_CALCULATE_CHI2 | mk.KFO_UPDATE_PARAMS
    ctx.propagate_helix_to_r(barrel["err"], barrel["par"], barrel["chg"], barrel["r"], e0, p0,
                             pflags=mk.PF_APPLY_MATERIAL, no_mat=barrel["no_mat"], out_fail=fail)
    ctx.kalman_operation(both, e0, p0, barrel["me"], barrel["mp"], ue0, up0, c0)
    ctx.propagate_helix_to_z(endcap["err"], endcap["par"], endcap["chg"], endcap["mp"][2], e1, p1)
    ctx.kalman_operation(both, e1, p1, endcap["me"], endcap["mp"], ue1, up1, c1, endcap=True)
    return [e0, p0, fail, ue0, up0, c0, e1, p1, ue1, up1, c1]


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "fit":
        slots, flop = {1: (17, FLOP_BARREL), 2: (25, FLOP_BARREL), 3: (15.4, 1240)}[case["geometry"]]
        return {"bytes": n * (slots * 37 + 232), "flops": n * slots * flop}
    if kind == "ops":
        return {"bytes": n * (2 * (27 + 1 + 1 + 27) + 2 * (27 + 9 + 28)) * 4, "flops": n * (FLOP_BARREL + FLOP_ENDCAP)}
    if kind == "find":
        L, area = (9, 2.0e5) if case["disks"] else (17, 8.2e4)
        seeds = n * case["events"]
        hits = case["events"] * L * (n + area * case["noise"])
        K = case["max_cands"]
        noise = (0.2 + 0.8 * case["noise"] / 2.0) * (0.4 + 0.1 * K if K > 1 else 1.0)
        return {"bytes": 36 * hits + seeds * (28 * 4 + 12 + K * (31 + L) * 4),
                "flops": seeds * L * FLOP_SEED_LAYER[case["finder"]] * noise}
    if kind == "layer":
        return {"bytes": n * ((27 + 2 + 27 + 27 + 18 + 10) * 4 + 8 * (36 + 48)), "flops": n * (1394 + 8 * 1161)}
    if kind == "bkfit":
        return {"bytes": n * (14 * 36 + 17 * 4 + 230), "flops": n * (14 * 1322 + 413)}
    word = 2 if case["fp64"] else 1
    return {"bytes": n * (25 * 36 + 28 * 4 + 4), "flops": n * 25 * 1394 * 5 * word}


# ---------------------------------------------------------------------------------------------------------
# The same formulas in 64 bits.  States are [n, 6] and [n, 6, 6]; constants hold the values of the 32-bit
# literals of the formulas' source (PropagationMPlex.icc, PropagationMPlex.cc, KalmanUtilsMPlex.cc).
# ---------------------------------------------------------------------------------------------------------

_F = lambda v: float(np.float32(v))
SOL, PI, TWO_PI = _F(0.299792458), _F(3.14159265358979323846), _F(6.28318530717958647692)
C2, C4, S3 = 0.5, _F(0.04166667), _F(0.16666667)


def _sincos4(x):
    x2 = x * x
    return x - S3 * x * x2, 1 - C2 * x2 + C4 * x2 * x2


def _field(param, z, r, bf):
    return (_F(-3.94991e-06) * z * z + _F(7.53701e-06) * z + _F(3.8114)) * (_F(2.43878e-11) * r * r + 1) if param else bf


def _squash(phi):
    phi = torch.where(phi >= PI, phi - TWO_PI, phi)
    return torch.where(phi < -PI, phi + TWO_PI, phi)


def _material(P, C, rad, xi, sign, barrel):
    """applyMaterialEffects; rad, xi per track."""
    pt = 1 / P[:, 3]
    th = P[:, 5]
    p = pt / torch.sin(th)
    p2 = p * p
    mpi, me, ion = _F(0.140), _F(0.0005), _F(16.0e-9 * 10.75)
    beta2 = p2 / (p2 + mpi * mpi)
    beta = beta2.sqrt()
    inv = p / pt if barrel else 1 / torch.cos(th).abs()
    rad0 = rad
    rad = rad * inv
    on = (rad0 >= 1e-13) & (rad >= 1e-13)
    safe = torch.where(on, rad, torch.ones_like(rad))
    msc = _F(0.0136) * (1 + _F(0.038) * safe.log()) / (beta * p)
    msc2 = msc * msc * safe
    g2 = (p2 + mpi * mpi) / (mpi * mpi)
    g = g2.sqrt()
    wmax = 2 * me * beta2 * g2 / (1 + 2 * g * me / mpi + me * me / (mpi * mpi))
    half = math.log(_F(28.816e-9) * math.sqrt(_F(2.33) * _F(0.498)) / ion) + (beta * g).log() - 0.5
    dedx = torch.where(beta < 1, 2 * (xi * inv * (0.5 * (2 * me * beta2 * g2 * wmax / (ion * ion)).log() - beta2 - half) / beta2),
                       torch.zeros_like(beta))
    dp = sign * dedx / beta
    zero = torch.zeros_like(dp)
    new = p / ((p + dp).clamp(min=_F(0.001)) * pt)
    P = torch.cat([P[:, :3], torch.where(on, new, P[:, 3])[:, None], P[:, 4:]], 1)
    diag = torch.stack([zero, zero, zero, torch.where(on, dp * dp / (p2 * pt * pt), zero), torch.where(on, msc2, zero),
                        torch.where(on, msc2, zero)], 1)
    return P, C + torch.diag_embed(diag)


def _lookup(grid, z, r):
    rl, xi = grid
    zb, rb = (z.abs() * 300 / 300).long(), (r * 120 / 120).long()
    ok = (zb >= 0) & (zb < 300) & (rb >= 0) & (rb < 120)
    i = zb.clamp(0, 299) * 120 + rb.clamp(0, 119)
    zero = torch.zeros_like(z)
    return torch.where(ok, rl[i], zero), torch.where(ok, xi[i], zero)


def _conj(J, C):
    return torch.bmm(torch.bmm(J, C), J.transpose(1, 2).contiguous())


def _to_r(P, C, chg, r, bf, param=False, mat=None):
    """propagateHelixToR: the new state and the failure mask (a failed track keeps its state).  mat(z, r): x/X0
    and xi of the step."""
    x0, y0, z0, ipt, phi, th = P.unbind(1)
    rr = torch.sqrt(x0 * x0 + y0 * y0)
    k = chg * 100 / (-SOL * _field(param, z0, rr, bf))
    pt = 1 / ipt
    cp, sp = phi.cos(), phi.sin()
    px, py = cp * pt, sp * pt
    zero = torch.zeros_like(x0)
    dx, dy, di, dphi, D = -x0 / rr, -y0 / rr, zero, zero, zero
    fail = torch.zeros_like(x0, dtype=torch.bool)
    x, y = x0, y0
    for i in range(5):
        rr = torch.sqrt(x * x + y * y)
        o = rr * pt / (px * x + py * y)
        bad = (o > 5) | (o < 0)
        fail = fail | bad
        d = torch.where(bad, zero, (r - rr) * o)
        D = D + d
        sh, ch = _sincos4(d * ipt / k * 0.5)
        ca, sa = 1 - 2 * sh * sh, 2 * sh * ch
        pxn, pyn = px * ca - py * sa, py * ca + px * sa
        if i < 4:
            w = torch.where((r - rr).abs() < _F(0.0001), 1 / rr, zero)
            gdot = x * pxn + y * pyn
            dx = dx - (x * w) * (1 - ipt * w * gdot)
            dy = dy - (y * w) * (1 - ipt * w * gdot)
            t = d / k * ipt
            di = di - k * (x * (px * ca * t - py * sa * t - py * ca - px * sa + py) +
                           y * (py * ca * t + px * sa * t - py * sa + px * ca - px)) * pt * w
            dphi = dphi + k * (x * (py * sa - px + px * ca) - y * (px * sa - py + py * ca)) * w
        x = x + 2 * k * sh * (px * ch - py * sh)
        y = y + 2 * k * sh * (py * ch + px * sh)
        px, py = pxn, pyn
    a = D * ipt / k
    ax, ay, ai, ap = dx * ipt / k, dy * ipt / k, (ipt * di + D) / k, dphi * ipt / k
    sa, ca = _sincos4(a)
    cc, ss = cp * ca - sp * sa, sp * ca + cp * sa
    kp = k * pt
    u = ipt * ai
    cot = th.cos() / th.sin()
    one = torch.ones_like(x)
    J = torch.stack([
        1 + kp * ax * cc, kp * ay * cc, zero, kp * pt * (cp * (u * ca - sa) + sp * (1 - ca - u * sa)),
        kp * (cp * ap * ca - sp * ap * sa - sp * sa + cp * ca - cp), zero,
        kp * ax * ss, 1 + kp * ay * ss, zero, kp * pt * (sp * (u * ca - sa) + cp * (u * sa - (1 - ca))),
        kp * (sp * ap * ca + cp * ap * sa + sp * ca + cp * sa - sp), zero,
        kp * cot * ax, kp * cot * ay, one, kp * cot * pt * (u - a), kp * cot * ap, -kp * a / (th.sin() * th.sin()),
        zero, zero, zero, one, zero, zero,
        ax, ay, zero, ai, 1 + ap, zero,
        zero, zero, zero, zero, zero, one], 1).view(-1, 6, 6)
    N = torch.stack([x, y, z0 + kp * a * cot, ipt, phi + a, th], 1)
    M = C
    if mat is not None:
        rad, xi = mat(N[:, 2], r)
        N, M = _material(N, M, rad, xi, torch.where(r > torch.sqrt(x0 * x0 + y0 * y0), one, -one), True)
    N = torch.cat([N[:, :4], _squash(N[:, 4])[:, None], N[:, 5:]], 1)
    M = _conj(J, M)
    f = fail[:, None]
    return torch.where(f, P, N), torch.where(f[:, :, None], C, M), fail


def _to_z(P, C, chg, z, bf, param=False, mat=None):
    """propagateHelixToZ."""
    x0, y0, z0, ipt, phi, th = P.unbind(1)
    k = chg * 100 / (-SOL * _field(param, z0, torch.sqrt(x0 * x0 + y0 * y0), bf))
    pt = 1 / ipt
    cp, sp, tan, ic2 = phi.cos(), phi.sin(), th.tan(), 1 / (th.cos() * th.cos())
    px, py = cp * pt, sp * pt
    dz = z - z0
    a = dz * tan * ipt / k
    sh, ch = _sincos4(a * 0.5)
    ca, sa = 1 - 2 * sh * sh, 2 * sh * ch
    v, w = px * ca - py * sa, py * ca + px * sa
    zero, one = torch.zeros_like(x0), torch.ones_like(x0)
    J = torch.stack([
        one, zero, -tan * ipt * v, k * pt * pt * (cp * (a * ca - sa) + sp * 2 * sh * (sh - a * ch)),
        -2 * k * pt * sh * (sp * ch + cp * sh), dz * ipt * v * ic2,
        zero, one, -tan * ipt * w, k * pt * pt * (sp * (a * ca - sa) - cp * 2 * sh * (sh - a * ch)),
        2 * k * pt * sh * (cp * ch - sp * sh), dz * ipt * w * ic2,
        zero, zero, zero, zero, zero, zero,
        zero, zero, zero, one, zero, zero,
        zero, zero, -ipt * tan / k, tan * dz / k, one, ipt * dz / k * ic2,
        zero, zero, zero, zero, zero, one], 1).view(-1, 6, 6)
    N = torch.stack([x0 + 2 * k * sh * (px * ch - py * sh), y0 + 2 * k * sh * (py * ch + px * sh), z, ipt, phi + a, th], 1)
    M = C
    if mat is not None:
        rad, xi = mat(z, torch.sqrt(N[:, 0] ** 2 + N[:, 1] ** 2))
        N, M = _material(N, M, rad, xi, torch.where(z.abs() > z0.abs(), one, -one), False)
    N = torch.cat([N[:, :4], _squash(N[:, 4])[:, None], N[:, 5:]], 1)
    return N, _conj(J, M)


def _update(P, C, mp, V, endcap):
    """kalmanOperation with both outputs; endcap: mask of tracks updated on a plane (x, y), the others on a cylinder
    (r-phi, z)."""
    n = P.shape[0]
    zero, one = torch.zeros_like(P[:, 0]), torch.ones_like(P[:, 0])
    r = torch.sqrt(mp[:, 0] ** 2 + mp[:, 1] ** 2)
    r = torch.where(endcap, one, r)
    a0, a1 = -(mp[:, 1] + P[:, 1]) / (2 * r), (mp[:, 0] + P[:, 0]) / (2 * r)
    h0 = torch.stack([torch.where(endcap, one, a0), torch.where(endcap, zero, a1), zero], 1)
    h1 = torch.stack([zero, torch.where(endcap, one, zero), torch.where(endcap, zero, one)], 1)
    H = torch.stack([h0, h1], 1)                                   # [n, 2, 3]
    HT = H.transpose(1, 2).contiguous()
    S = torch.bmm(torch.bmm(H, C[:, :3, :3] + V), HT)
    det = S[:, 0, 0] * S[:, 1, 1] - S[:, 0, 1] * S[:, 1, 0]
    I = torch.stack([S[:, 1, 1] / det, -S[:, 0, 1] / det, -S[:, 1, 0] / det, S[:, 0, 0] / det], 1).view(n, 2, 2)
    res = torch.bmm(H, (mp - P[:, :3])[:, :, None])
    chi2 = torch.bmm(torch.bmm(res.transpose(1, 2).contiguous(), I), res)[:, 0, 0]
    K = torch.bmm(torch.bmm(C[:, :, :3].contiguous(), HT), I)
    N = P + torch.bmm(K, res)[:, :, 0]
    N = torch.cat([N[:, :4], _squash(N[:, 4])[:, None], N[:, 5:]], 1)
    M = C - torch.bmm(K, torch.bmm(H, C[:, :3, :].contiguous()))
    return N, (M + M.transpose(1, 2)) / 2, chi2


_TRI = [(i, j) for i in range(6) for j in range(i + 1)]


def _full(packed, size=6):
    """[..packed.., n] lower triangle to [n, size, size]."""
    out = torch.zeros(packed.shape[-1], size, size, dtype=torch.float64, device=packed.device)
    for e, (i, j) in enumerate(t for t in _TRI if t[0] < size):
        out[:, i, j] = out[:, j, i] = packed[e].double()
    return out


def _packed(C):
    return torch.stack([C[:, i, j] for i, j in _TRI])


def _pca_z(P):
    t = P[:, 5].tan()
    return t * (t * P[:, 2] - torch.sqrt(P[:, 0] ** 2 + P[:, 1] ** 2)) / (1 + t * t)


def _grid(geo):
    return tuple(_gpu(g.reshape(-1)).double() for g in mk.material_grid(geo))


def _step(P, C, chg, mp, V, real, endcap, bf, param=False, grid=None, fake_mat=False):
    """One hit slot of a fit: a track without a hit of its own (not `real`) takes a wide one at its position."""
    mp = torch.where(real[:, None], mp, P[:, :3])
    V = torch.where(real[:, None, None], V, torch.eye(3, dtype=V.dtype, device=V.device) * 666.0)
    mat = None
    if grid is not None:
        def mat(z, r):
            rad, xi = _lookup(grid, z, r)
            off = torch.zeros_like(rad)
            return (rad, xi) if fake_mat else (torch.where(real, rad, off), torch.where(real, xi, off))
    r = torch.sqrt(mp[:, 0] ** 2 + mp[:, 1] ** 2)
    PB, CB, _ = _to_r(P, C, chg, r, bf, param, mat)
    if bool(endcap.any()):
        PZ, CZ = _to_z(P, C, chg, mp[:, 2], bf, param, mat)
        PB, CB = torch.where(endcap[:, None], PZ, PB), torch.where(endcap[:, None, None], CZ, CB)
    return _update(PB, CB, mp, V, endcap)


def _exact_fit(case, seed):
    geo, ev = _fit_tracks(case, seed)
    grid, bf = _grid(geo), _F(BFIELD)
    P, C, chg = ev["seed_par"].double().T.contiguous(), _full(ev["seed_err"]), ev["chg"].double()
    chi2 = torch.zeros_like(chg)
    for s in range(ev["hit_pos"].shape[0]):
        at = (s < ev["n_hits"]).nonzero()[:, 0]
        if not len(at):
            break
        fl = ev["hit_flags"][s, at]
        N, M, c2 = _step(P[at], C[at], chg[at], ev["hit_pos"][s][:, at].double().T.contiguous(),
                         _full(ev["hit_err"][s][:, at], 3), (fl & mk.HIT_MISSING) == 0, (fl & mk.HIT_ENDCAP) != 0, bf,
                         grid=grid)
        q = chg[at]
        if case["pca"]:
            flip = N[:, 3] < 0
            q = torch.where(flip, -q, q)
            N[:, 3] = N[:, 3].abs()
        P[at], C[at], chg[at] = N, M, q
        chi2[at] += c2
    if case["pca"]:
        P, C = _to_z(P, C, chg, _pca_z(P), bf)
    return [P.T, _packed(C), None, chi2]


def _exact_ops(case, seed):
    geo, ev = _barrel_tracks(case["n"], seed)
    disk = _disk_tracks(case["n"], seed)
    grid, bf, n = _grid(geo), _F(BFIELD), case["n"]
    none, every = torch.zeros(n, dtype=torch.bool, device=DEV), torch.ones(n, dtype=torch.bool, device=DEV)
    with_mat = _no_material(ev) == 0
    mp, r = ev["hit_pos"][1], torch.hypot(ev["hit_pos"][1, 0], ev["hit_pos"][1, 1]).double()
    off = torch.zeros_like(r)
    P, C, _ = _to_r(ev["seed_par"].double().T.contiguous(), _full(ev["seed_err"]), ev["chg"].double(), r, bf,
                    mat=lambda z, rr: tuple(torch.where(with_mat, v, off) for v in _lookup(grid, z, rr)))
    UP, UC, c0 = _update(P, C, mp.double().T.contiguous(), _full(ev["hit_err"][1], 3), none)
    mz = disk["hit_pos"][1].double().T.contiguous()
    Q, D = _to_z(disk["seed_par"].double().T.contiguous(), _full(disk["seed_err"]), disk["chg"].double(), mz[:, 2].clone(), bf)
    UQ, UD, c1 = _update(Q, D, mz, _full(disk["hit_err"][1], 3), every)
    return [_packed(C), P.T, None, _packed(UC), UP.T, c0, _packed(D), Q.T, _packed(UD), UQ.T, c1]


def _exact_bkfit(case, seed):
    geo, offset, hits, cand, base = _bk_inputs(case, seed)
    L, n, G = geo.n_barrel, case["n"], case["group"]
    offset = torch.from_numpy(offset.astype(np.int64)).to(DEV)
    P, C, chg = cand["par"].double().T.contiguous(), _full(cand["err"] * 100.0), cand["chg"].double()
    chi2 = torch.zeros_like(chg)
    block = torch.arange(n, device=DEV) // G
    for l in range(L - 1, -1, -1):
        h = cand["hot_idx"][l].long()
        has = h >= 0
        some = torch.zeros(int(block[-1]) + 1, dtype=torch.bool, device=DEV)
        some[block[has]] = True
        at = some[block].nonzero()[:, 0]
        if not len(at):
            continue
        hh = hits[(offset[base.long()[at] + l] + h[at].clamp(min=0)).clamp(max=hits.shape[0] - 1)]
        N, M, c2 = _step(P[at], C[at], chg[at], hh[:, :3].double(), _full(hh[:, 3:].T, 3), has[at],
                         torch.zeros(len(at), dtype=torch.bool, device=DEV), 0.0, param=True)
        flip = N[:, 3] < 0
        chg[at] = torch.where(flip, -chg[at], chg[at])
        N[:, 3] = N[:, 3].abs()
        P[at], C[at] = N, M
        chi2[at] += c2
    if case["pca"]:
        P, C = _to_z(P, C, chg, _pca_z(P), 0.0, param=True)
    found = (cand["hot_idx"] >= 0).sum(0).double()
    behind = (cand["hot_idx"] >= 0).flip(0).cumsum(0).flip(0) > 0       # a hit on this layer or one after it
    holes = ((cand["hot_idx"] == -1) & behind).sum(0).double()
    low = (1 / P[:, 3]).abs() < _F(0.9)
    bonus = _F(0.2) * found + 4.0
    bonus = torch.where(low, bonus.clamp(max=8.0), bonus)
    score = bonus * found - torch.where(low, 12.0, 8.0) * holes - chi2.clamp(min=0)
    return [P.T, _packed(C), None, chi2, score]


def _exact_adjoint(case, seed):
    ev, theta = _adjoint_inputs(case, seed)
    th = _gpu(theta).double().requires_grad_(True)
    bf, xi_per_x0 = _F(BFIELD), _F(2.2e-3)
    chi2, grads = [], torch.zeros_like(th)
    for lo in range(0, case["n"], 25_000):
        sl = slice(lo, min(case["n"], lo + 25_000))
        P, C, chg = ev["seed_par"][:, sl].double().T.contiguous(), _full(ev["seed_err"][:, sl]), ev["chg"][sl].double()
        tot = torch.zeros_like(chg)
        barrel = torch.zeros(len(chg), dtype=torch.bool, device=DEV)
        for l in range(ev["hit_pos"].shape[0]):
            on = l < ev["n_hits"][sl]
            hp = ev["hit_pos"][l][:, sl].double()
            x = torch.where(on, hp[0], torch.ones_like(hp[0]))           # unused slots hold zeros
            y = torch.where(on, hp[1], torch.zeros_like(hp[1]))
            ir = 1 / torch.sqrt(x * x + y * y)
            mp = torch.stack([x - th[l, 1] * (y * ir), y + th[l, 1] * (x * ir), hp[2] + th[l, 2]], 1)
            r = torch.sqrt(mp[:, 0] ** 2 + mp[:, 1] ** 2)
            rad = th[l, 0].expand(len(chg))
            N, M, _ = _to_r(P, C, chg, r, bf, mat=lambda z, rr: (rad, rad * xi_per_x0))
            V = _full(ev["hit_err"][l][:, sl], 3)
            V = torch.where(on[:, None, None], V, torch.eye(3, dtype=V.dtype, device=DEV))
            N, M, c2 = _update(N, M, mp, V, barrel)
            P, C = torch.where(on[:, None], N, P), torch.where(on[:, None, None], M, C)
            tot = tot + torch.where(on, c2, torch.zeros_like(c2))
        grads += torch.autograd.grad(tot.sum(), th)[0]
        chi2.append(tot.detach())
    return [torch.cat(chi2), grads]


def exact(case, seed):
    """What `run` returns, in 64 bits.  The finders and the layer step have no such value: which hits they take,
    and with them every number that follows, is decided by comparisons of 32-bit values."""
    f = {"fit": _exact_fit, "ops": _exact_ops, "bkfit": _exact_bkfit, "adjoint": _exact_adjoint}.get(case["kind"])
    return None if f is None else f(case, seed)
