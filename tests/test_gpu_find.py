"""GPU parity of best-hit finding: the HIP LayerOfHits build, SelectHitIndices and the fused
FindTracksBestHit loop (through the C ABI) against the CPU oracle on the same toy events.

Integer results (hit ranks, bin ranges, candidate lists, chosen hit indices) must agree exactly
except where a float32 rounding difference decides a comparison: a hit on a bin or window edge, or
two candidates whose chi2 agree to rounding.  Those cases are counted and bounded explicitly.
"""
import numpy as np
import pytest

import mkfit_amd as mk
import oracle
from _common import RawDeviceBuffer, par_rel
from _find_common import (F_PHI_FINE, _brute_select, _keys, _random_hits, assert_bins, assert_find_parity,
                          best_hit_reference, edge_explained, pad_seed_hits)

pytestmark = pytest.mark.gpu


def _t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def _event(seed, n_tracks, noise, pt_min=0.5):
    geo = mk.geometry(1)
    p = mk.default_toy_params(seed=seed, simulate_material=0, pt_min=pt_min, pt_max=10.0)
    ev = mk.generate_find_event(geo, p, n_tracks, noise_per_cm2=noise)
    return geo, ev, mk.barrel_layer_descs(geo)


@pytest.fixture(scope="module")
def setup(gpu_device):
    geo, ev, descs = _event(123, 5000, 3.0)
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, descs)
    hits = _t(ev["hits_flat"], gpu_device)
    eoh.load(ev["hit_offset"], hits)
    return ev, descs, ctx, eoh


def _fine_boundary(phi):
    """phi within a few ulps of a fine phi-bin edge (one ulp of phi moves the scaled value by ~4e-5)."""
    x = F_PHI_FINE * (phi + np.float32(np.pi))
    return np.abs(x - np.round(x)) < 3e-4


def test_loh_build_matches_oracle(setup):
    ev, descs, ctx, eoh = setup
    off = ev["hit_offset"]
    flips = 0
    for l in range(len(descs)):
        hl = ev["hits_flat"][off[l]:off[l + 1]]
        r_c, b_c, p_c, q_c, nq_c = oracle.loh_build(descs[l], hl)
        r_g, b_g, p_g, q_g, nq_g = eoh.layer_views(l)
        assert nq_g == nq_c and len(r_g) == len(hl)
        assert sorted(r_g.tolist()) == list(range(len(hl)))
        # per original hit: phi to an ulp (device vs host atan2f), q exact
        phi_c = np.empty_like(p_c); phi_c[r_c] = p_c
        phi_g = np.empty_like(p_g); phi_g[r_g] = p_g
        q_o = np.empty_like(q_g); q_o[r_g] = q_g
        assert np.array_equal(q_o, hl[:, 2])
        # device and host atan2f agree to a few ulp (both within their documented error bounds)
        dphi = np.abs(phi_g - phi_c)
        dphi = np.minimum(dphi, np.abs(dphi - np.float32(2 * np.pi)))
        assert np.all(dphi <= 4 * np.spacing(np.maximum(np.abs(phi_c), np.float32(1e-6)))), dphi.max()
        k_c, _ = _keys(descs[l], phi_c, hl[:, 2])
        k_g, _ = _keys(descs[l], phi_g, hl[:, 2])
        moved = k_c != k_g
        assert np.all(_fine_boundary(phi_c[moved])), "a key differs away from a bin edge"
        flips += int(moved.sum())
        if not moved.any():
            assert np.array_equal(r_g, r_c), l
            assert_bins(b_g, b_c, l)
        else:
            assert np.array_equal(np.argsort(k_g, kind="stable"), r_g)
    # a hit lands within a few ulp of one of the 1024 fine-bin edges with probability ~1e-4, and the two
    # atan2f implementations then disagree on the bin about a third of the time
    assert flips <= max(5, 1e-4 * off[-1]), (flips, off[-1])


def _crowded_event(descs, seed=5):
    """Hits of four barrel layers piled into few (q, fine phi) bins, in shuffled order: 10,000 copies of one
    hit (beyond the LDS sort), 3,000 of another (sorted in LDS), 150 positions x 40 copies (one thread's
    share exceeded many times), and hits at phi = +pi exactly (fine bin 1024, sorting last in its q row but
    filling coarse bin 0) and -pi, each layer with random hits among them."""
    rng = np.random.default_rng(seed)

    def hit(r, phi, z):
        return [r * np.cos(phi), r * np.sin(phi), z, 1e-4, 0.0, 1e-4, 0.0, 0.0, 1e-2]

    def rand(d, n):
        return [hit(d["propagate_to"], rng.uniform(-np.pi, np.pi), rng.uniform(d["zmin"], d["zmax"]))
                for _ in range(n)]
    layers = []
    d = descs[0]
    layers.append([hit(d["propagate_to"], 0.3, 1.0)] * 10000 + rand(d, 500))
    d = descs[1]
    layers.append([hit(d["propagate_to"], -2.0, -3.0)] * 3000 + rand(d, 200))
    d = descs[2]
    pos = [(rng.uniform(-np.pi, np.pi), rng.uniform(d["zmin"], d["zmax"])) for _ in range(150)]
    layers.append([hit(d["propagate_to"], p, z) for p, z in pos for _ in range(40)] + rand(d, 100))
    d = descs[3]
    r = d["propagate_to"]
    plus = [[-r, 0.0, 2.0, 1e-4, 0.0, 1e-4, 0.0, 0.0, 1e-2]] * 50          # atan2(+0, -r) = +pi
    minus = [[-r, -0.0, 2.0, 1e-4, 0.0, 1e-4, 0.0, 0.0, 1e-2]] * 50        # atan2(-0, -r) = -pi
    near = [hit(r, -np.pi + 1e-3, 2.0)] * 30                                # coarse bin 0 of the same row
    layers.append(plus + minus + near + rand(d, 100))
    out = []
    for h in layers:
        h = np.array(h, np.float32)
        out.append(h[rng.permutation(len(h))])
    return out


def test_loh_crowded_bins(gpu_device):
    """The LayerOfHits build keeps the reference's stable order and bin ranges however the hits crowd."""
    geo = mk.geometry(1)
    descs = mk.barrel_layer_descs(geo)[:4]
    layers = _crowded_event(descs)
    off = np.concatenate([[0], np.cumsum([len(h) for h in layers])]).astype(np.int32)
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, descs)
    eoh.load(off, _t(np.concatenate(layers), gpu_device))
    for l, hl in enumerate(layers):
        r_c, b_c, p_c, q_c, nq_c = oracle.loh_build(descs[l], hl)
        r_g, b_g, p_g, q_g, nq_g = eoh.layer_views(l)
        phi_c = np.empty_like(p_c); phi_c[r_c] = p_c
        phi_g = np.empty_like(p_g); phi_g[r_g] = p_g
        k_c, _ = _keys(descs[l], phi_c, hl[:, 2])
        k_g, _ = _keys(descs[l], phi_g, hl[:, 2])
        assert np.array_equal(np.argsort(k_g, kind="stable"), r_g), l
        if np.array_equal(k_c, k_g):
            assert np.array_equal(r_g, r_c), l
            assert_bins(b_g, b_c, l)
        else:
            assert np.all(_fine_boundary(phi_c[k_c != k_g])), l
    # fine bin 1024: the +pi hits own coarse bin 0 of their q row, after the row's other hits
    r_g, b_g, p_g, _, _ = eoh.layer_views(3)
    assert np.sum(p_g == np.float32(np.pi)) == 50
    ctx.close()


def test_loh_reload_smaller_event(setup, gpu_device):
    ev, descs, ctx, eoh = setup
    geo, ev2, _ = _event(7, 300, 0.5)
    e2 = mk.EventOfHits(ctx, descs)
    e2.load(ev["hit_offset"], _t(ev["hits_flat"], gpu_device))     # large first, then the small one
    e2.load(ev2["hit_offset"], _t(ev2["hits_flat"], gpu_device))
    off = ev2["hit_offset"]
    for l in (0, 7, 16):
        hl = ev2["hits_flat"][off[l]:off[l + 1]]
        r_c, b_c, p_c, _, _ = oracle.loh_build(descs[l], hl)
        r_g, b_g, p_g, _, _ = e2.layer_views(l)
        # the layer holds exactly the small event's hits, ordered by the device's own keys
        assert sorted(r_g.tolist()) == list(range(len(hl)))
        phi_g = np.empty_like(p_g); phi_g[r_g] = p_g
        k_g, _ = _keys(descs[l], phi_g, hl[:, 2])
        assert np.array_equal(np.argsort(k_g, kind="stable"), r_g)
        phi_c = np.empty_like(p_c); phi_c[r_c] = p_c
        k_c, _ = _keys(descs[l], phi_c, hl[:, 2])
        if np.array_equal(k_g, k_c):            # no fine-bin flip: identical to the oracle
            assert_bins(b_g, b_c)
            assert np.array_equal(r_g, r_c)


def _random_states(rng, n, r, zspan):
    par = np.zeros((6, n), np.float32); err = np.zeros((21, n), np.float32)
    phi = rng.uniform(-np.pi, np.pi, n).astype(np.float32)
    par[0] = r * np.cos(phi); par[1] = r * np.sin(phi); par[2] = rng.uniform(-zspan, zspan, n)
    par[3] = rng.uniform(0.1, 2, n); par[4] = phi; par[5] = rng.uniform(0.3, 2.8, n)
    s = rng.uniform(1e-4, 0.3, n).astype(np.float32) ** 2
    err[0] = s; err[2] = s; err[1] = rng.uniform(-0.5, 0.5, n) * s; err[5] = rng.uniform(1e-4, 0.8, n) ** 2
    return par, err


@pytest.mark.parametrize("layer", [3, 9, 16])
def test_select_hit_indices_matches_oracle(setup, gpu_device, layer):
    import torch
    ev, descs, ctx, eoh = setup
    d = descs[layer]
    off = ev["hit_offset"]
    hl = ev["hits_flat"][off[layer]:off[layer + 1]]
    rng = np.random.default_rng(layer)
    n = 4000
    par, err = _random_states(rng, n, d["propagate_to"], d["zmax"] + 1.5)
    xs = torch.zeros(n, dtype=torch.int32, device=gpu_device)
    xa = torch.zeros((16, n), dtype=torch.int32, device=gpu_device)
    w = torch.zeros(n, dtype=torch.int32, device=gpu_device)
    eoh.select_hit_indices(layer, _t(par, gpu_device), _t(err, gpu_device), xs, xa, w)
    xs, xa, w = xs.cpu().numpy(), xa.cpu().numpy(), w.cpu().numpy()
    xs_c, xa_c, w_c = oracle.select_hit_indices(d, hl, par, err)
    wsr_diff = np.nonzero(w != w_c)[0]
    assert len(wsr_diff) <= 2
    ranks, _, phis, qs, _ = oracle.loh_build(d, hl)
    same = (xs == xs_c) & np.all(xa == xa_c, axis=0)
    bad = np.nonzero(~same & (w == w_c))[0]
    if len(bad):
        _, wins = _brute_select(d, hl, par[:, bad], err[:, bad], ranks, phis, qs)
        for k, t in enumerate(bad):
            diff = np.setxor1d(xa[:max(xs[t], 0), t], xa_c[:max(xs_c[t], 0), t])
            assert edge_explained(wins[k], par[:, t], hl, diff), (t, xa[:, t], xa_c[:, t])
    assert len(bad) <= n // 500
    assert (xs == 16).sum() > 0 and (xs == -1).sum() > 0 and (xs == 0).sum() > 0


def _run_find(ctx, eoh, ev, n_layers, first_layer, dev, chi2_cut=15.0):
    import torch
    b = mk.FindBatch(ev, n_layers, first_layer, device=dev, chi2_cut=chi2_cut)
    ctx.find_tracks_best_hit(eoh, b)
    torch.cuda.synchronize()
    return b, b.numpy()


def _compare_find(gpu, ev, descs, first_layer=3, **kw):
    """The GPU's best-hit result against the oracle's, seed by seed (assert_find_parity); returns the oracle's."""
    cpu, spread = best_hit_reference(ev, descs, first_layer, n_threads=8, bfield=3.8, **kw)
    assert_find_parity("best hit", gpu, cpu, spread, first_layer)
    return cpu


def _true_fraction(res, ev, first_layer):
    hot = res["hot_idx"][first_layer:]
    off = ev["hit_offset"][first_layer:-1]
    ok = hot >= 0
    truth = np.where(ok, ev["hit_mc"][off[:, None] + np.maximum(hot, 0)], -5)
    return (truth == ev["seed_mc"][None, :]).sum() / hot.size


def test_find_best_hit_matches_oracle(setup, gpu_device):
    ev, descs, ctx, eoh = setup
    _, gpu = _run_find(ctx, eoh, ev, len(descs), 3, gpu_device)
    cpu = _compare_find(gpu, ev, descs, chi2_cut=15.0)
    assert abs(_true_fraction(gpu, ev, 3) - _true_fraction(cpu, ev, 3)) < 2e-3
    assert _true_fraction(gpu, ev, 3) > 0.8


def test_find_best_hit_propagate_to_hit(setup, gpu_device):
    import torch
    ev, descs, ctx, eoh = setup
    b = mk.FindBatch(ev, len(descs), 3, device=gpu_device, chi2_cut=15.0, prop_to_hit=True)
    ctx.find_tracks_best_hit(eoh, b)
    torch.cuda.synchronize()
    _compare_find(b.numpy(), ev, descs, chi2_cut=15.0, prop_to_hit=True)


def test_find_noise_free_exact_path(gpu_device):
    geo, ev, descs = _event(31, 3000, 0.0, pt_min=1.0)
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, descs)
    eoh.load(ev["hit_offset"], _t(ev["hits_flat"], gpu_device))
    _, gpu = _run_find(ctx, eoh, ev, len(descs), 3, gpu_device)
    _compare_find(gpu, ev, descs)
    assert _true_fraction(gpu, ev, 3) > 0.97


def test_find_repeatable(setup, gpu_device):
    ev, descs, ctx, eoh = setup
    b, r1 = _run_find(ctx, eoh, ev, len(descs), 3, gpu_device)
    b.reset()
    ctx.find_tracks_best_hit(eoh, b)
    r2 = b.numpy()
    for k in r1:
        assert np.array_equal(r1[k], r2[k]), k


def test_find_edge_cases(setup, gpu_device):
    import torch
    ev, descs, ctx, eoh = setup
    L = len(descs)
    # nothing to search: the seeds come back unchanged
    b, g = _run_find(ctx, eoh, pad_seed_hits(ev, L), L, L, gpu_device)
    assert np.array_equal(g["par"], ev["seed_par"]) and np.array_equal(g["hot_idx"][:3], ev["seed_hits"][:3])
    assert np.all(g["hot_idx"][3:] == -1)
    assert np.array_equal(g["n_found"], np.sum(ev["seed_hits"] >= 0, axis=0))
    # no seeds
    e0 = dict(ev, n_seeds=0)
    b0 = mk.FindBatch(e0, L, 3, device=gpu_device)
    ctx.find_tracks_best_hit(eoh, b0)
    # empty layers 5 and 6, then an event without hits at all
    off = ev["hit_offset"]
    keep = np.ones(off[-1], bool); keep[off[5]:off[7]] = False
    cnt = np.diff(off).copy(); cnt[5] = cnt[6] = 0
    ev2 = dict(ev, hits_flat=ev["hits_flat"][keep], hit_offset=np.concatenate([[0], np.cumsum(cnt)]).astype(np.int32),
               hit_mc=ev["hit_mc"][keep])
    for evx in (ev2, dict(ev, hits_flat=np.zeros((0, 9), np.float32), hit_offset=np.zeros(L + 1, np.int32),
                          hit_mc=np.zeros(0, np.int32))):
        ex = mk.EventOfHits(ctx, descs)
        ex.load(evx["hit_offset"], _t(evx["hits_flat"], gpu_device) if len(evx["hits_flat"]) else
                torch.zeros((1, 9), device=gpu_device))
        _, g = _run_find(ctx, ex, evx, L, 3, gpu_device)
        _compare_find(g, evx, descs)
        assert np.all(g["hot_idx"][5:7] < 0)


def test_find_rejects_bad_arguments(setup, gpu_device):
    import torch
    ev, descs, ctx, eoh = setup
    b = mk.FindBatch(ev, len(descs), 3, device=gpu_device)
    b.first_layer = len(descs) + 1
    with pytest.raises(mk.MkfError, match="first_layer"):
        ctx.find_tracks_best_hit(eoh, b)
    b = mk.FindBatch(ev, len(descs), 3, device=gpu_device)
    with RawDeviceBuffer(2 * b.n * 4) as short:                  # too short for 17 layers
        b.hot_idx = short
        with pytest.raises(mk.MkfError, match="hot_idx"):
            ctx.find_tracks_best_hit(eoh, b)
    fresh = mk.EventOfHits(ctx, descs)
    with pytest.raises(mk.MkfError, match="not loaded"):
        ctx.find_tracks_best_hit(fresh, mk.FindBatch(ev, len(descs), 3, device=gpu_device))
    with pytest.raises(mk.MkfError, match="hit_offset"):
        fresh.load(np.array([0, 5, 3] + [3] * (len(descs) - 2), np.int32), torch.zeros((5, 9), device=gpu_device))


def test_find_on_endcap_disks(gpu_device):
    geo = mk.geometry(4)
    p = mk.default_toy_params(seed=14, simulate_material=0, eta_max=2.5, pt_min=1.0)
    ev = mk.generate_find_event(geo, p, 4000, noise_per_cm2=1.0)
    descs = mk.disk_layer_descs(geo)
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, descs)
    eoh.load(ev["hit_offset"], _t(ev["hits_flat"], gpu_device))
    for l in (0, 4, 8):
        r_c, b_c, _, _, _ = oracle.loh_build(descs[l], ev["hits_flat"][ev["hit_offset"][l]:ev["hit_offset"][l + 1]])
        r_g, b_g, _, _, _ = eoh.layer_views(l)
        assert np.mean(r_g == r_c) > 0.999
    _, gpu = _run_find(ctx, eoh, ev, len(descs), 3, gpu_device)
    _compare_find(gpu, ev, descs, chi2_cut=15.0)



def test_hit_mask_matches_oracle(gpu_device):
    """The iteration's hit mask (mkf_event_of_hits_set_hit_mask): best-hit and clone-engine finding with 40 %
    of the finding layers' hits masked match the oracle run with the same mask, seed by seed; clearing the
    mask and a new load give the unmasked result back bit for bit."""
    import torch
    from _find_common import assert_ce_parity, clone_engine_reference
    geo, ev, descs = _event(9, 3000, 2.0)
    rng = np.random.default_rng(9)
    total = int(ev["hit_offset"][-1])
    mask = (rng.random(total) < 0.4).astype(np.uint8)
    mask[:ev["hit_offset"][3]] = 0
    evm = dict(ev, hit_mask=mask)
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, descs)
    eoh.load(ev["hit_offset"], _t(ev["hits_flat"], gpu_device))

    def run_bh():
        b = mk.FindBatch(ev, len(descs), 3, device=gpu_device, chi2_cut=15.0)
        ctx.find_tracks_best_hit(eoh, b)
        torch.cuda.synchronize()
        return b.numpy()

    def run_ce():
        c = mk.CEBatch(ev, len(descs), 3, device=gpu_device, chi2_cut=30.0, max_cands=6)
        ctx.find_tracks_clone_engine(eoh, c)
        torch.cuda.synchronize()
        return c.numpy()
    plain_bh, plain_ce = run_bh(), run_ce()
    eoh.set_hit_mask(_t(mask, gpu_device))
    bh, ce = run_bh(), run_ce()
    off = ev["hit_offset"]
    for l in range(3, len(descs)):
        for h in (bh["hot_idx"][l], ce["hot_idx"][:, l]):
            assert not mask[h[h >= 0] + off[l]].any(), l
    _compare_find(bh, evm, descs, chi2_cut=15.0)
    cpu, spread = clone_engine_reference(evm, descs, 3, chi2_cut=30.0, max_cands=6, n_threads=8)
    assert_ce_parity("masked clone engine", ce, cpu, spread, 3)
    eoh.set_hit_mask(None)
    for a, b in ((run_bh(), plain_bh), (run_ce(), plain_ce)):
        for k in a:
            assert np.array_equal(a[k], b[k]), k
    eoh.set_hit_mask(_t(mask, gpu_device))
    eoh.load(ev["hit_offset"], _t(ev["hits_flat"], gpu_device))
    a = run_bh()
    for k in a:
        assert np.array_equal(a[k], plain_bh[k]), k
    ctx.close()


def _rows_of_keys(key, nq):
    """Bin ranges of a layer from its hits' keys, as LayerOfHits::SuckInHits leaves them: the phi == +pi run
    (fine bin 1024) of a row overwrites coarse bin 0."""
    ks = np.sort(key)
    bins = np.zeros((nq * 256, 2), np.int64)
    for q in range(nq):
        edge = np.searchsorted(ks, (q << 16) + np.append(np.arange(0, 1024, 4), [1024, 1025]))
        for b in range(256):
            if edge[b] < edge[b + 1]:
                bins[q * 256 + b] = edge[b], edge[b + 1]
        if edge[256] < edge[257]:
            bins[q * 256] = edge[256], edge[257]
    return bins


@pytest.mark.parametrize("q_bin,is_barrel", [(0.15, 1), (2.0, 1), (30.0, 1), (120.0, 1), (1.5, 0), (60.0, 0)])
def test_loh_order_for_row_and_tile_sizes(gpu_device, q_bin, is_barrel):
    """Sizes around the tile and row capacity (3072 hits) and one hit or none, from 800 q bins down to one: rows
    sorted in one go, in runs, and by several blocks."""
    import torch
    rng = np.random.default_rng(int(q_bin * 100) + is_barrel)
    sizes = [0, 1, 3071, 3072, 3073, 0, 9000, 40000, 2]
    descs, hits = [], []
    for n in sizes:
        r = 20.0 if is_barrel else rng.uniform(2.0, 55.0, n)
        phi = rng.uniform(-np.pi, np.pi, n)
        z = rng.uniform(-62.0, 62.0, n) if is_barrel else np.full(n, 30.0)
        if n > 1000:
            phi[:200] = np.pi                              # fine bin 1024
            phi[200:600] = phi[600]                        # one crowded fine bin
        h = np.zeros((n, 9), np.float32)
        h[:, 0], h[:, 1], h[:, 2] = r * np.cos(phi), r * np.sin(phi), z
        h[:200, 1] = np.where(np.arange(len(h[:200])) % 2 == 0, 0.0, h[:200, 1]) if n > 1000 else h[:200, 1]
        h[:, 3:] = rng.uniform(0.0, 1.0, (n, 6))
        hits.append(h[rng.permutation(n)] if n > 1000 else h)
        descs.append(dict(is_barrel=is_barrel, rin=2.0 if not is_barrel else 19.99, rout=50.0 if not is_barrel else 20.01,
                          zmin=-60.0 if is_barrel else 29.99, zmax=60.0 if is_barrel else 30.01,
                          propagate_to=20.0 if is_barrel else 30.0, q_bin=q_bin, min_dphi=0.002, max_dphi=0.1, min_dq=0.3,
                          max_dq=2.0, c_dp_sf=1.1, c_dq_sf=1.1, c_c2_sf=1.1))
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    flat = np.concatenate(hits)
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, descs)
    eoh.load(off, torch.from_numpy(flat).to(gpu_device))
    for l, h in enumerate(hits):
        _check_layer_of_hits(ctx, eoh, l, descs[l], h, gpu_device)
    # the mask in sorted order: with every hit masked but one, a search around it finds that one
    last = sizes.index(9000)
    h = hits[last]
    q = h[:, 2] if is_barrel else np.hypot(h[:, 0], h[:, 1])
    keep = int(np.nonzero(np.abs(q - (0.0 if is_barrel else 25.0)) < 20.0)[0][3])
    x, y, z = h[keep, :3]
    mask = np.ones(off[-1], np.uint8)
    mask[off[last] + keep] = 0
    eoh.set_hit_mask(torch.from_numpy(mask).to(gpu_device))
    par = np.array([[x], [y], [z], [0.5], [np.arctan2(y, x)], [1.2]], np.float32)
    err = np.zeros((21, 1), np.float32)
    err[[0, 2, 5, 9, 14, 20], 0] = 1e-4
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu_device)
    xs, xa, w = t(np.zeros(1, np.int32)), t(np.zeros((16, 1), np.int32)), t(np.zeros(1, np.int32))
    eoh.select_hit_indices(last, t(par), t(err), xs, xa, w)
    assert xs.item() == 1 and xa[0, 0].item() == keep
    eoh.close()
    ctx.close()


def test_loh_order_beyond_the_tile_table(gpu_device):
    """A layer of more tiles (261 of 3072 hits) than a row's block keeps, beside a small one."""
    import torch
    rng = np.random.default_rng(77)
    d = dict(is_barrel=1, rin=19.99, rout=20.01, zmin=-60.0, zmax=60.0, propagate_to=20.0, q_bin=0.5, min_dphi=0.002,
             max_dphi=0.1, min_dq=0.3, max_dq=2.0, c_dp_sf=1.1, c_dq_sf=1.1, c_c2_sf=1.1)
    n = 800_000
    phi, z = rng.uniform(-np.pi, np.pi, n + 10), rng.uniform(-60.0, 60.0, n + 10)
    h = np.zeros((n + 10, 9), np.float32)
    h[:, 0], h[:, 1], h[:, 2] = 20 * np.cos(phi), 20 * np.sin(phi), z
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, [d, d])
    eoh.load(np.array([0, n, n + 10], np.int32), torch.from_numpy(h).to(gpu_device))
    for l, hl in ((0, h[:n]), (1, h[n:])):
        ranks, bins, phis, qs, nq = eoh.layer_views(l)
        ph = np.arctan2(hl[:, 1].astype(np.float64), hl[:, 0].astype(np.float64)).astype(np.float32)
        lo, extent = np.float32(-60.0), np.float32(120.0)
        extra = np.float32(0.5) * (np.float32(nq) * np.float32(0.5) - extent)
        qb = np.clip(((hl[:, 2] - (lo - extra)) * (np.float32(nq) / extent)).astype(np.int64), 0, nq - 1)
        key = np.floor(F_PHI_FINE * (ph + np.float32(np.pi))).astype(np.int64) + (qb << 16)
        assert np.array_equal(ranks, np.argsort(key, kind="stable"))
        assert np.array_equal(phis, ph[ranks]) and np.array_equal(qs, hl[ranks, 2])
        want = _rows_of_keys(key, nq)
        full = want[:, 0] < want[:, 1]
        assert np.array_equal(bins[full], want[full])
    eoh.close()
    ctx.close()


def _repeat(ev, times):
    """The event with its seeds repeated: every copy must come out as the first."""
    out = dict(ev, n_seeds=ev["n_seeds"] * times)
    for k in ("seed_par", "seed_err", "seed_chg", "seed_hits"):
        out[k] = np.concatenate([ev[k]] * times, axis=-1)
    return out


def _first(ev, n):
    return dict(ev, n_seeds=n, **{k: np.ascontiguousarray(ev[k][..., :n])
                                  for k in ("seed_par", "seed_err", "seed_chg", "seed_hits")})


@pytest.mark.parametrize("prop_to_hit", [False, True])
def test_best_hit_for_every_packing(setup, gpu_device, prop_to_hit):
    """Seeds per wavefront follow the batch size (1 to 64): the tracks do not depend on it."""
    ev, descs, ctx, eoh = setup
    ev = _first(ev, 1100)

    def run(e):
        b = mk.FindBatch(e, len(descs), 3, device=gpu_device, chi2_cut=15.0, prop_to_hit=prop_to_hit)
        ctx.find_tracks_best_hit(eoh, b)
        return b.numpy()
    whole = run(ev)
    for n in (1, 63, 1025):
        part = run(_first(ev, n))
        assert all(np.array_equal(part[k], whole[k][..., :n], equal_nan=True) for k in whole), n
    for times in (2, 5, 16, 61):                     # 2 .. 64 seeds per wavefront, the last wavefront part filled
        many = run(_repeat(ev, times))
        for k in whole:
            assert np.array_equal(many[k], np.concatenate([whole[k]] * times, axis=-1), equal_nan=True), (times, k)


@pytest.mark.parametrize("finder,max_cands", [("ce", 1), ("ce", 6), ("ce", 8), ("std", 3), ("std", 8)])
def test_combinatorial_for_every_packing(setup, gpu_device, finder, max_cands):
    """Seeds per wavefront follow the batch size (1 to 10, or 8 slots' 8): the candidates do not depend on it."""
    ev, descs, ctx, eoh = setup
    ev = _first(ev, 900)

    def run(e):
        b = mk.CEBatch(e, len(descs), 3, device=gpu_device, chi2_cut=30.0, max_cands=max_cands)
        (ctx.find_tracks_clone_engine if finder == "ce" else ctx.find_tracks_standard)(eoh, b)
        return b.numpy()
    whole = run(ev)
    part = run(_first(ev, 1))
    assert all(np.array_equal(part[k], whole[k][..., :1], equal_nan=True) for k in whole)
    for times in (5, 9, 27):
        many = run(_repeat(ev, times))
        for k in whole:
            assert np.array_equal(many[k], np.concatenate([whole[k]] * times, axis=-1), equal_nan=True), (times, k)


@pytest.mark.parametrize("min_dphi,min_dq", [(0.01, 1.0), (0.3, 2.0), (1.6, 9.0), (3.1, 300.0)])
def test_select_for_every_packing_and_window(gpu_device, min_dphi, min_dq):
    """Windows of one bin to the whole layer (several runs per q row across phi = +-pi, more rows than are read
    together, more chunks than the work list holds), for 1 to 64 windows per wavefront, against the oracle."""
    import torch
    rng = np.random.default_rng(31)
    d = dict(is_barrel=1, rin=19.99, rout=20.01, zmin=-60.0, zmax=60.0, propagate_to=20.0, q_bin=2.0, min_dphi=min_dphi,
             max_dphi=3.14, min_dq=min_dq, max_dq=400.0, c_dp_sf=1.1, c_dq_sf=1.1, c_c2_sf=1.1)
    n_hits, n = 12000, 70000
    phi, z = rng.uniform(-np.pi, np.pi, n_hits), rng.uniform(-60.0, 60.0, n_hits)
    h = np.zeros((n_hits, 9), np.float32)
    h[:, 0], h[:, 1], h[:, 2], h[:, 3], h[:, 5], h[:, 8] = 20 * np.cos(phi), 20 * np.sin(phi), z, 1e-4, 1e-4, 1e-2
    tp = np.where(rng.random(n) < 0.3, np.pi - rng.uniform(0, 0.05, n), rng.uniform(-np.pi, np.pi, n))
    par = np.stack([20 * np.cos(tp), 20 * np.sin(tp), rng.uniform(-62.0, 62.0, n), np.full(n, 0.5), tp,
                    rng.uniform(0.6, 2.5, n)]).astype(np.float32)
    err = np.zeros((21, n), np.float32)
    err[[0, 2, 5, 9, 14, 20]] = 1e-4
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, [d])
    eoh.load(np.array([0, n_hits], np.int32), torch.from_numpy(h).to(gpu_device))

    def run(m):
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu_device)
        xs, xa, w = t(np.zeros(m, np.int32)), t(np.zeros((16, m), np.int32)), t(np.zeros(m, np.int32))
        eoh.select_hit_indices(0, t(par[:, :m]), t(err[:, :m]), xs, xa, w)
        return xs.cpu().numpy(), xa.cpu().numpy(), w.cpu().numpy()
    whole = run(n)
    for m in (1, 3, 700, 1025, 9001, 40000):
        assert all(np.array_equal(a, b[..., :m]) for a, b in zip(run(m), whole)), m
    m = 400
    xs, xa, w = oracle.select_hit_indices(d, h, np.ascontiguousarray(par[:, :m]), np.ascontiguousarray(err[:, :m]))
    # one float rounding of a bin or window edge moves a lane's list: at most a lane in a hundred
    same = (xs == whole[0][:m]) & (w == whole[2][:m])
    for k in range(m):
        same[k] &= np.array_equal(xa[:max(xs[k], 0), k], whole[1][:max(xs[k], 0), k])
    assert same.mean() >= 0.99, same.mean()
    eoh.close()
    ctx.close()


def _one_layer(n_hits, rng, min_dphi, min_dq):
    d = dict(is_barrel=1, rin=19.99, rout=20.01, zmin=-60.0, zmax=60.0, propagate_to=20.0, q_bin=2.0, min_dphi=min_dphi,
             max_dphi=3.14, min_dq=min_dq, max_dq=400.0, c_dp_sf=1.1, c_dq_sf=1.1, c_c2_sf=1.1)
    phi, z = rng.uniform(-np.pi, np.pi, n_hits), rng.uniform(-60.0, 60.0, n_hits)
    h = np.zeros((n_hits, 9), np.float32)
    h[:, 0], h[:, 1], h[:, 2], h[:, 3], h[:, 5], h[:, 8] = 20 * np.cos(phi), 20 * np.sin(phi), z, 1e-4, 1e-4, 1e-2
    return d, h


def _tracks(n, rng):
    tp = rng.uniform(-np.pi, np.pi, n)
    par = np.stack([20 * np.cos(tp), 20 * np.sin(tp), rng.uniform(-58.0, 58.0, n), np.full(n, 0.5), tp,
                    rng.uniform(0.6, 2.5, n)]).astype(np.float32)
    err = np.zeros((21, n), np.float32)
    err[[0, 2, 5, 9, 14, 20]] = 1e-4
    return par, err


@pytest.mark.parametrize("min_dphi,min_dq,free", [(3.1, 300.0, 0.0002), (3.1, 300.0, 0.002), (0.3, 3.0, 0.01),
                                                  (0.3, 3.0, 0.1), (1.0, 25.0, 0.0)])
def test_select_in_windows_of_many_masked_hits(gpu_device, min_dphi, min_dq, free):
    """Windows of many hits, nearly all of them masked, so that a list fills late or never, scanned by the wavefront
    or, where it holds too many, by lane; plain windows and ones of many rows; against the oracle."""
    import torch
    rng = np.random.default_rng(int(min_dq * 10 + free * 1e4))
    d, h = _one_layer(60000, rng, min_dphi, min_dq)
    mask = (rng.random(len(h)) >= free).astype(np.uint8)
    n = 4000
    par, err = _tracks(n, rng)
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, [d])
    eoh.load(np.array([0, len(h)], np.int32), torch.from_numpy(h).to(gpu_device))
    eoh.set_hit_mask(torch.from_numpy(mask).to(gpu_device))
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu_device)

    def run(m, times=1):
        xs, xa, w = (t(np.zeros(m * times, np.int32)), t(np.zeros((16, m * times), np.int32)),
                     t(np.zeros(m * times, np.int32)))
        eoh.select_hit_indices(0, t(np.tile(par[:, :m], times)), t(np.tile(err[:, :m], times)), xs, xa, w)
        return xs.cpu().numpy(), xa.cpu().numpy(), w.cpu().numpy()
    whole = run(n)
    for m in (1, 5, 900):
        assert all(np.array_equal(a, b[..., :m]) for a, b in zip(run(m), whole)), m
    for a, b in zip(run(n, 17), whole):
        assert np.array_equal(a, np.concatenate([b] * 17, axis=-1))
    m = 300
    xs, xa, w = oracle.select_hit_indices(d, h, np.ascontiguousarray(par[:, :m]), np.ascontiguousarray(err[:, :m]), mask)
    # one float rounding of a bin or window edge moves a lane's list: at most a lane in a hundred
    same = (xs == whole[0][:m]) & (w == whole[2][:m])
    for k in range(m):
        same[k] &= np.array_equal(xa[:max(xs[k], 0), k], whole[1][:max(xs[k], 0), k])
    assert same.mean() >= 0.99, same.mean()
    eoh.close()
    ctx.close()


@pytest.mark.parametrize("n", [1, 1000, 70000])
def test_wide_windows_cost_what_sixteen_hits_cost(gpu_device, n):
    """A list is full at 16 hits: windows over a whole layer of 50k hits take a few times as long as ordinary ones
    (reading all of every window took a hundred to ten thousand times as long)."""
    import torch
    took = []
    for min_dphi, min_dq in ((0.01, 1.0), (3.1, 300.0)):
        rng = np.random.default_rng(5)
        d, h = _one_layer(50000, rng, min_dphi, min_dq)
        par, err = _tracks(n, rng)
        ctx = mk.Context(bfield=3.8)
        eoh = mk.EventOfHits(ctx, [d])
        eoh.load(np.array([0, len(h)], np.int32), torch.from_numpy(h).to(gpu_device))
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu_device)
        a = [t(par), t(err), t(np.zeros(n, np.int32)), t(np.zeros((16, n), np.int32)), t(np.zeros(n, np.int32))]
        times = []
        for _ in range(7):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            eoh.select_hit_indices(0, *a)
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1))
        took.append(float(np.median(times)))
        eoh.close()
        ctx.close()
    assert took[1] < 20 * took[0], took


def _layer_desc(q_bin=0.5, is_barrel=1):
    return dict(is_barrel=is_barrel, rin=19.99 if is_barrel else 2.0, rout=20.01 if is_barrel else 50.0,
                zmin=-60.0 if is_barrel else 29.99, zmax=60.0 if is_barrel else 30.01,
                propagate_to=20.0 if is_barrel else 30.0, q_bin=q_bin, min_dphi=0.002, max_dphi=0.1, min_dq=0.3,
                max_dq=2.0, c_dp_sf=1.1, c_dq_sf=1.1, c_c2_sf=1.1)


def _hits_at(phi, q, rng, is_barrel=1):
    """Hits of a layer at phi and q (z, or r on a disk), in random order, each with its own covariance."""
    n = len(phi)
    r = 20.0 if is_barrel else q
    h = np.zeros((n, 9), np.float32)
    h[:, 0], h[:, 1], h[:, 2] = r * np.cos(phi), r * np.sin(phi), q if is_barrel else 30.0
    h[phi == np.pi, 1] = 0.0                               # phi of the stored hit is +pi itself
    h[:, 3], h[:, 5], h[:, 8] = rng.uniform(1e-4, 1e-2, (3, n))
    return h[rng.permutation(n)]


def _check_layer_of_hits(ctx, eoh, l, d, h, dev):
    """Everything a load leaves of layer l: order, phi, q, bin ranges, and, hit by hit through the inverse map, the
    sorted copies (an update with the loaded hit against the same update from the event of hits)."""
    import torch
    ranks, bins, phis, qs, nq = eoh.layer_views(l)
    phi = np.arctan2(h[:, 1].astype(np.float64), h[:, 0].astype(np.float64)).astype(np.float32)
    assert np.array_equal(np.sort(ranks), np.arange(len(h)))
    assert np.array_equal(phis, phi[ranks])
    q = np.empty_like(qs)
    q[ranks] = qs
    r2 = h[:, 0].astype(np.float64) ** 2 + h[:, 1].astype(np.float64) ** 2
    assert np.array_equal(q, h[:, 2]) if d["is_barrel"] else np.allclose(q, np.sqrt(r2), rtol=2e-7, atol=0)
    lo, hi = (np.float32(d[k]) for k in (("zmin", "zmax") if d["is_barrel"] else ("rin", "rout")))
    extra = np.float32(0.5) * (np.float32(nq) * np.float32(d["q_bin"]) - (hi - lo))
    qb = np.clip(((q - (lo - extra)) * (np.float32(nq) / (hi - lo))).astype(np.int64), 0, nq - 1)
    key = np.floor(F_PHI_FINE * (phi + np.float32(np.pi))).astype(np.int64) + (qb << 16)
    assert np.array_equal(ranks, np.argsort(key, kind="stable"))
    want = _rows_of_keys(key, nq)
    full = want[:, 0] < want[:, 1]
    assert np.array_equal(bins[full], want[full]) and np.all(bins[~full, 0] == bins[~full, 1])
    n = len(h)
    if n == 0:
        return key
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    par = np.tile(np.array([[20.0], [0.5], [1.0], [0.5], [0.1], [1.4]], np.float32), n)
    err = np.zeros((21, n), np.float32)
    err[[0, 2, 5, 9, 14, 20]] = np.array([100.0, 80.0, 60.0, 1e-4, 1e-3, 1e-3], np.float32)[:, None]
    err[1], err[3], err[4] = 5.0, 3.0, -2.0
    lanes = mk.FinderLanes(t(par), t(err), t(np.ones(n, np.int32)))
    ctx.update_with_last_hit(eoh, l, lanes, t(np.arange(n, dtype=np.int32)), prop_to_hit=False)
    out_err, out_par = t(np.zeros_like(err)), t(np.zeros_like(par))
    ctx.kalman_operation(2, t(err), t(par), t(h[:, 3:].T), t(h[:, :3].T), out_err, out_par, endcap=not d["is_barrel"])
    got = lanes.numpy()
    # the same arithmetic in two kernels, whose fused operations may round differently
    assert np.allclose(got["par"], out_par.cpu().numpy(), rtol=1e-5, atol=1e-4)
    assert np.allclose(got["err"], out_err.cpu().numpy(), rtol=1e-4, atol=1e-4)
    return key


@pytest.mark.parametrize("is_barrel", [1, 0])
def test_loh_order_of_full_rows_and_crowded_bins(gpu_device, is_barrel):
    """Rows and fine phi bins around and beyond what one block orders: whole rows of 3071 to 20000 hits, one fine bin of
    256, 257, 3072 and 7000 hits over several tiles with others before and after it, runs at phi = +pi, a layer in
    one q bin, and layers in one fine bin."""
    import torch
    rng = np.random.default_rng(91 + is_barrel)
    u = lambda n: rng.uniform(-np.pi, np.pi, n)
    qmid = 10.25
    spread = lambda n: rng.uniform(3.0, 49.0, n)
    layers = []
    for n in (3071, 3072, 3073, 6145, 20000):               # one full row among others
        layers.append((np.concatenate([u(n), u(5000)]), np.concatenate([np.full(n, qmid), spread(5000)])))
    for n in (256, 257, 3072, 7000):                        # one crowded fine bin, in a row of others
        layers.append((np.concatenate([rng.uniform(0.501, 0.502, n), u(1500), u(9000)]),
                       np.concatenate([np.full(n + 1500, qmid), spread(9000)])))
    for n in (1, 257, 4000):                                # phi = +pi, alone in its row and not
        layers.append((np.concatenate([np.full(n, np.pi), u(4000)]), np.concatenate([np.full(n, qmid), spread(4000)])))
        layers.append((np.concatenate([np.full(n, np.pi), u(700), u(9)]),
                       np.concatenate([np.full(n + 700, qmid), spread(9)])))
    layers.append((u(9000), np.full(9000, qmid)))           # one q bin
    for n in (256, 257, 3072, 3073, 12000):                 # one fine bin, and nothing else
        layers.append((rng.uniform(0.501, 0.502, n), np.full(n, qmid)))
    layers.append((u(40), spread(40)))
    d = _layer_desc(is_barrel=is_barrel)
    hits = [_hits_at(phi, q, rng, is_barrel) for phi, q in layers]
    off = np.concatenate([[0], np.cumsum([len(h) for h in hits])]).astype(np.int32)
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, [d] * len(hits))
    flat = torch.from_numpy(np.concatenate(hits)).to(gpu_device)
    for _ in range(2):                                      # a second load finds the first one's tables
        eoh.load(off, flat)
        crowd = 0
        for l, h in enumerate(hits):
            key = _check_layer_of_hits(ctx, eoh, l, d, h, gpu_device)
            crowd = max(crowd, np.bincount(key).max())
        assert crowd >= 12000
    eoh.close()
    ctx.close()


def test_loh_order_beyond_four_million_hits(gpu_device):
    """Loads whose sorted copies are stored past the caches, with even layers, a skewed one and one in one fine bin."""
    import torch
    rng = np.random.default_rng(92)
    d, n = _layer_desc(), 170_000
    hits = [_hits_at(rng.uniform(-np.pi, np.pi, n), rng.uniform(-60.0, 60.0, n), rng) for _ in range(4)]
    hits.append(_hits_at(rng.uniform(-np.pi, np.pi, n), rng.uniform(3.0, 4.0, n), rng))
    hits.append(_hits_at(rng.uniform(0.501, 0.502, n), np.full(n, 7.1), rng))
    copies = 26
    order = [l % len(hits) for l in range(copies)]
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, [d] * copies)
    dev = [torch.from_numpy(h).to(gpu_device) for h in hits]
    eoh.load((np.arange(copies + 1) * n).astype(np.int32), torch.cat([dev[i] for i in order]))
    for l in (0, 3, 4, 5, 20, 23, 25):
        _check_layer_of_hits(ctx, eoh, l, d, hits[order[l]], gpu_device)
    eoh.close()
    ctx.close()


def test_loh_order_of_a_layer_of_millions(gpu_device):
    """Above 2^21 hits in a layer the load goes through the radix sort; just below, through the rows."""
    import torch
    rng = np.random.default_rng(94)
    d = _layer_desc(q_bin=2.0)
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, [d, d])
    for n in ((1 << 21) + 1, 1 << 21):
        hits = [_hits_at(rng.uniform(-np.pi, np.pi, m), np.where(rng.random(m) < 0.3, 7.1, rng.uniform(-60.0, 60.0, m)),
                         rng) for m in (n, 5000)]
        eoh.load(np.array([0, n, n + 5000], np.int32), torch.from_numpy(np.concatenate(hits)).to(gpu_device))
        for l in (0, 1):
            _check_layer_of_hits(ctx, eoh, l, d, hits[l], gpu_device)
    eoh.close()
    ctx.close()


def test_captured_load_sorts_what_the_buffer_holds(gpu_device):
    """A load recorded in a graph and replayed on other hits of the same number: which rows are put off is decided on the
    device, replay by replay."""
    import torch
    rng = np.random.default_rng(95)
    d, n = _layer_desc(), 15000
    u = lambda: rng.uniform(-np.pi, np.pi, n)
    kinds = [(u(), rng.uniform(-60.0, 60.0, n)), (u(), np.full(n, 3.1)), (rng.uniform(0.501, 0.502, n), np.full(n, 3.1)),
             (u(), rng.uniform(-60.0, 60.0, n))]
    hits = [_hits_at(phi, q, rng) for phi, q in kinds]
    ctx = mk.Context(bfield=3.8)
    eoh = mk.EventOfHits(ctx, [d, d])
    off = np.array([0, n, 2 * n], np.int32)
    buf = torch.from_numpy(np.concatenate([hits[0], hits[0]])).to(gpu_device)
    eoh.load(off, buf)                       # allocates
    torch.cuda.synchronize()
    g, st = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(g, stream=st):
        eoh.load(off, buf)
    for a, b in ((1, 0), (2, 1), (0, 3), (3, 2)):
        buf.copy_(torch.from_numpy(np.concatenate([hits[a], hits[b]])).to(gpu_device))
        g.replay()
        torch.cuda.synchronize()
        _check_layer_of_hits(ctx, eoh, 0, d, hits[a], gpu_device)
        _check_layer_of_hits(ctx, eoh, 1, d, hits[b], gpu_device)
    del g
    eoh.close()
    ctx.close()


def test_load_time_does_not_depend_on_the_distribution(gpu_device):
    """Hits crowded into two q bins, into one, or into one fine bin load within a few times an even layer's time (one
    block per full row took up to a thousand times as long)."""
    import torch
    rng = np.random.default_rng(93)
    n, d = 150_000, _layer_desc()
    u = lambda: rng.uniform(-np.pi, np.pi, n)
    kinds = [(u(), rng.uniform(-60.0, 60.0, n)), (u(), rng.uniform(3.0, 4.0, n)), (u(), np.full(n, 3.1)),
             (rng.uniform(0.501, 0.502, n), np.full(n, 3.1))]
    ctx = mk.Context(bfield=3.8)
    took = []
    for phi, q in kinds:
        h = torch.from_numpy(_hits_at(phi, q, rng)).to(gpu_device).repeat(4, 1)
        eoh = mk.EventOfHits(ctx, [d] * 4)
        off = (np.arange(5) * n).astype(np.int32)
        times = []
        for _ in range(7):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            eoh.load(off, h)
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1))
        took.append(float(np.median(times)))
        eoh.close()
    assert max(took) < 10 * took[0], took
    ctx.close()
