"""GPU parity of the reconstruction path (libbsx through the C-ABI) against the
FP64 CPU oracle on the same seeded inputs.

Tolerances (from the reconstruction target): finished map FSC >= 0.9999 in
every shell and max |gpu - oracle| / max |oracle| <= 1e-4; accumulators within
FP32 accumulation error (1e-4 relative to the plane maximum; the reference
also accumulates in FP32)."""
import math
import sys

import numpy as np
import pytest
import torch

from bsoft_amd import abi, synth
from bsoft_amd.abi import BsxError, ReconParams
from bsoft_amd.recon import Reconstruction, part_ft_size, symmetry_views
from oracle.oracle import Oracle, OracleRecon

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def dataset(n_map, nblobs, nparts, box, seed, snr=0.1, defocus=(1e4, 3e4), astig=(0.0, 0.0)):
    rng = np.random.default_rng(seed)
    bm = synth.make_blob_map(n_map, nblobs, rng)
    ps = synth.make_particles(bm, nparts, box, rng, snr=snr, defocus=defocus, astig=astig, seed=seed)
    return bm, ps


def run_pair(ps, *, size, box, ft, interp=0, ctf=1, flags=0, nhalves=1, wiener=0.2, hi_res=1.5,
             imap=0, nmaps=1, npartial=2, batch=0, lo_res=0.0):
    say(f"case size={size} box={box} ft={ft} interp={interp} ctf={ctf} flags={flags} "
        f"nhalves={nhalves} nmaps={nmaps}/{imap} n={len(ps.parts)}")
    dev_imgs = ps.images.to("cuda").contiguous()
    rec = Reconstruction(size, box, ft, 1.5, hi_res=hi_res, lo_res=lo_res, interp=interp,
                         ctf_action=ctf, wiener=wiener, flags=flags, nhalves=nhalves, batch=batch)
    rec.insert(dev_imgs, ps.parts)
    g = rec.finish(imap, nmaps, want_ft=True, want_fom=bool(flags & abi.BSX_FLAG_FOM))
    torch.cuda.synchronize()
    rp = ReconParams(size=size, box=box, ft_size=ft, interp=interp, sampling=1.5, hi_res=hi_res,
                     lo_res=lo_res, ctf_action=ctf, flags=flags & ~abi.BSX_FLAG_TIMING,
                     wiener=wiener, nhalves=nhalves, batch=0, mem_cap=0)
    o = OracleRecon(rp, npartial, 64)
    o.insert(synth.particles_list(ps.parts), ps.images.cpu().numpy())
    m, fom, ftc, st = o.finish(imap, nmaps, want_ft=True, want_fom=bool(flags & abi.BSX_FLAG_FOM))
    return rec, g, (m, fom, ftc, st), o


def check_map(g, ref, fsc_min=0.9999, rel=1e-4):
    m, _, ftc, st = ref
    gm = g.map.cpu().numpy().astype(np.float64)
    err = np.abs(gm - m).max() / np.abs(m).max()
    f, sup = Oracle(64).fsc_with_support(g.ft.cpu().numpy(), ftc, 1.5, 1.5)
    say(f"  max rel err {err:.3e}  min FSC {f[sup].min():.6f} over {sup.sum()}/{len(f)} shells"
        f"  coverage {g.coverage}/{st.coverage}")
    assert err <= rel
    assert f[sup].min() >= fsc_min
    assert np.all(f[1:][~sup[1:]] == 0)          # shell 0 is set to 1 by definition
    assert g.coverage == st.coverage
    # Friedel residual (absolute amplitude units, as friedel_check prints it)
    # FP32 rounding leaves a residual of order 1e-7 of the amplitude scale
    assert abs(g.friedel - st.friedel) <= 1e-3 * st.friedel + 1e-5 * np.abs(ftc).max()
    assert g.particles == st.particles
    return err, f


def test_c1_full_config_flip():
    """The CPU-runnable configuration in full: 64^3 map of 40 blobs, 2000
    particles at uniform views, CTF 300 kV / Cs 2.7 mm / amp 0.07, defocus
    U[1,3] um, SNR 0.1, NN insertion, pad 2 (ft 128), CTF flip."""
    bm, ps = dataset(64, 40, 2000, 64, seed=0)
    rec, g, ref, o = run_pair(ps, size=64, box=64, ft=128)
    check_map(g, ref)
    acc = rec.accumulators(0).cpu().numpy().astype(np.float64)
    oa = sum(o.partial_acc(t) for t in range(o.T))
    for q, tol in [(0, 1e-4), (1, 1e-4), (2, 1e-4)]:
        e = np.abs(acc[q] - oa[q]).max() / np.abs(oa[q]).max()
        say(f"  plane {q} rel err {e:.3e}")
        assert e <= tol
    # weights: every one of the ft^2 samples is inserted with w = 1/(0.6*4)
    assert acc[2].sum() == pytest.approx(2000 * 128 * 128 / 2.4, rel=1e-5)


@pytest.mark.parametrize("interp", [1, 2])
def test_interpolation_modes(interp):
    bm, ps = dataset(32, 10, 300, 32, seed=1)
    rec, g, ref, _ = run_pair(ps, size=32, box=32, ft=64, interp=interp)
    check_map(g, ref)


@pytest.mark.parametrize("ctf,wiener", [(0, 0.0), (2, 0.0), (4, 0.2), (4, 0.05), (2, 0.3),
                                        (7, 0.2)])
def test_ctf_actions(ctf, wiener):
    bm, ps = dataset(32, 10, 300, 32, seed=2, astig=(0.0, 2000.0))
    rec, g, ref, _ = run_pair(ps, size=32, box=32, ft=64, ctf=ctf, wiener=wiener)
    check_map(g, ref)


def _fom_conditioning(planes, hmask):
    """Per voxel, how much the SNR figure of merit's numerator W |F|^2 - P
    cancels (fspace_reconstruction_snr, Bimage_reconstruct.cpp:610-634, on
    the values fspace_reconstruction_weigh leaves): |W|F|^2| / |W|F|^2 - P|.
    Used only to pick the voxels where FP32 inputs fix the FOM to ~1e-5."""
    acc = sum(planes[h].astype(np.float64) for h in range(len(planes)) if (hmask >> h) & 1)
    fr, fi, W, P, W2 = acc
    ok = W > 1e-30
    Ws = np.where(ok, W, 1.0)
    sig = (fr / Ws) ** 2 + (fi / Ws) ** 2
    w2 = Ws - W2 / Ws
    Pn = np.where(w2 > 1, P / np.where(w2 > 1, w2, 1), np.where(Ws > 1, P / Ws, P))
    Pn = np.maximum(Pn, 0)
    num = Ws * sig - Pn
    return np.where(ok & (Ws > 1), np.abs(Ws * sig) / np.maximum(np.abs(num), 1e-300), np.inf)


def test_half_maps_and_fom():
    """Half maps and the SNR figure of merit. The FOM is checked twice, both
    times by its maximum error: against the FP64 oracle's finish of the GPU's
    own accumulator sums (the weighing and FOM formulas alone, every voxel
    whose numerator cancels by less than 100x), and against the oracle's own
    reconstruction (accumulation order included) on the same voxels."""
    bm, ps = dataset(32, 10, 400, 32, seed=3)
    for imap, nmaps in [(0, 2), (1, 2), (0, 3), (2, 3)]:
        rec, g, ref, o = run_pair(ps, size=32, box=32, ft=64, nhalves=2, nmaps=nmaps, imap=imap,
                                  flags=abi.BSX_FLAG_FOM)
        check_map(g, ref)
        gf = g.fom.cpu().numpy().astype(np.float64)
        planes = [rec.accumulators(h).cpu().numpy() for h in range(2)]
        own = OracleRecon(o.rp, 2, 64)
        for h in range(2):
            own.set_partial_acc(h, planes[h])
        _, fom_own, _, _ = own.finish(imap, nmaps, want_fom=True)
        hmask = 3
        if nmaps == 2:
            hmask = 1 << (imap % 2)
        if nmaps == 3 and imap % 3:
            hmask = 1 << (imap % 3 - 1)
        cond = _fom_conditioning(planes, hmask)
        sel = (cond < 100) & (np.abs(fom_own) > 1e-6)
        sel.flat[0] = False                      # FOM[0] is set to 1
        e_own = np.max(np.abs(gf[sel] - fom_own[sel]) / np.abs(fom_own[sel]))
        of = ref[1]
        sel2 = sel & (np.abs(of) > 1e-6)
        e_ref = np.max(np.abs(gf[sel2] - of[sel2]) / np.abs(of[sel2]))
        say(f"  FOM: max rel err {e_own:.2e} vs FP64 finish of the same sums, {e_ref:.2e} vs the "
            f"oracle's reconstruction, over {sel.sum()} of {gf.size} voxels")
        assert sel.sum() > 0.2 * gf.size
        assert e_own <= 1e-4
        assert e_ref <= 1e-3
        # voxels with a weight sum of at most 1 have FOM 0 (:624)
        W = sum(planes[h][2].astype(np.float64) for h in range(2) if (hmask >> h) & 1)
        low = W <= 1
        low.flat[0] = False
        assert np.all(gf[low] == 0)


def test_ewald_mag_lowres_bootstrap():
    bm, ps = dataset(32, 10, 200, 32, seed=4)
    rng = np.random.default_rng(4)
    ps.parts["mag"] = rng.uniform(0.95, 1.05, len(ps.parts))
    ps.parts["sel"] = rng.integers(1, 4, len(ps.parts))
    ps.parts["ori"] += rng.uniform(-2, 2, (len(ps.parts), 2))
    rec, g, ref, _ = run_pair(ps, size=32, box=32, ft=64,
                              flags=abi.BSX_FLAG_EWALD | abi.BSX_FLAG_BOOTSTRAP, lo_res=40.0,
                              hi_res=4.0)
    check_map(g, ref)


def test_box_smaller_than_map_pad3():
    """Map 48^3 from 40^2 particles, pad 3 (ft 128): size/box mismatch and a
    map edge that needs a radix-3 inverse FFT."""
    bm, ps = dataset(48, 10, 150, 40, seed=5)
    ft = part_ft_size(48, 1, 3)
    assert ft == 256
    rec, g, ref, _ = run_pair(ps, size=48, box=40, ft=128)
    check_map(g, ref)


def test_batching_is_invisible():
    bm, ps = dataset(32, 10, 100, 32, seed=6)
    d = ps.images.cuda()
    r1 = Reconstruction(32, 32, 64, 1.5, ctf_action=1, batch=7)
    r1.insert(d, ps.parts)
    r2 = Reconstruction(32, 32, 64, 1.5, ctf_action=1, batch=1000)
    r2.insert(d[:40].contiguous(), ps.parts[:40])
    r2.insert(d[40:].contiguous(), ps.parts[40:])
    a1, a2 = r1.accumulators(0), r2.accumulators(0)
    assert torch.allclose(a1[2], a2[2], rtol=1e-5, atol=1e-5)
    assert (a1[:3] - a2[:3]).abs().max() <= 1e-5 * a1[:3].abs().max()


def test_c2_shape_properties():
    """256^3 map from 256^2 particles (ft 512) with astigmatism: size-independent
    properties — weight total, Friedel symmetry — and oracle parity on a
    subset small enough for the CPU."""
    bm, ps = dataset(256, 400, 64, 256, seed=7, snr=0.05, defocus=(8e3, 3.5e4), astig=(0, 2000))
    d = ps.images.cuda()
    rec = Reconstruction(256, 256, 512, 1.5, ctf_action=1)
    rec.insert(d, ps.parts)
    g = rec.finish(want_ft=True)
    assert g.weight_sum == pytest.approx(64 * 512 * 512 / 2.4, rel=1e-6)
    assert math.isfinite(g.friedel)
    sub = synth.ParticleSet(images=ps.images[:6].contiguous(), parts=ps.parts[:6].copy())
    rec2, g2, ref, _ = run_pair(sub, size=256, box=256, ft=512)
    check_map(g2, ref)


def test_empty_and_errors():
    rec = Reconstruction(32, 32, 64, 1.5, ctf_action=1, flags=abi.BSX_FLAG_CHECK_NAN)
    rec.insert(torch.empty((0, 32, 32), device="cuda"), np.zeros(0, dtype=synth.PARTICLE_DTYPE))
    g = rec.finish()
    assert g.coverage == 0 and g.particles == 0
    assert torch.all(g.map == 0)
    bm, ps = dataset(32, 4, 4, 32, seed=8)
    imgs = ps.images.clone()
    imgs[2, 5, 5] = float("nan")
    with pytest.raises(BsxError) as e:
        rec.insert(imgs.cuda(), ps.parts)
    assert e.value.code == abi.BSX_ERR_NONFINITE
    with pytest.raises(BsxError) as e:
        Reconstruction(256, 256, 512, 1.5, mem_cap=64 << 20)
    assert e.value.code == abi.BSX_ERR_NOMEM
    with pytest.raises(BsxError) as e:
        rec.finish(1, 2)      # half map from a single accumulator
    assert e.value.code == abi.BSX_ERR_STATE
    bad = ps.parts.copy()
    bad["pixel_size"][1] = 0
    with pytest.raises(BsxError):
        rec.insert(ps.images.cuda(), bad)


@pytest.mark.parametrize("interp", [0, 1, 2])
@pytest.mark.parametrize("ft,n", [(128, 64), (64, 32), (512, 128)])
def test_variants_agree(interp, ft, n):
    """XCD accumulator copies, orientation ordering and run merging change only
    the FP32 summation order: every variant matches the plain path."""
    say(f"variants interp={interp} ft={ft} n={n}")
    bm, ps = dataset(n, 10, 60, n, seed=9)
    d = ps.images.cuda()
    ref = Reconstruction(n, n, ft, 1.5, ctf_action=1, interp=interp, method=1, order=1, merge=2)
    ref.insert(d, ps.parts)
    a0 = ref.accumulators(0)
    for method, order, merge, batch in [(0, 0, 1, 0), (0, 2, 1, 7), (0, 1, 2, 0), (1, 0, 1, 0)]:
        r = Reconstruction(n, n, ft, 1.5, ctf_action=1, interp=interp, method=method, order=order,
                           merge=merge, batch=batch)
        r.insert(d, ps.parts)
        a = r.accumulators(0)
        for q in range(3):
            e = ((a[q] - a0[q]).abs().max() / a0[q].abs().max()).item()
            assert e < 2e-5, (method, order, merge, q, e)


@pytest.mark.parametrize("interp", [0, 1, 2])
def test_fom_sums_binned_match_direct(interp):
    """With BSX_FLAG_FOM the binned insertion carries sum w|F|^2 and sum w^2
    of every entry in a second pool array and folds them with the Friedel-pair
    entries: all five accumulator planes of both half sets match the
    direct-atomic path (method 1) to FP32 summation order, and so do the FOM
    maps of the finish."""
    say(f"FOM binned vs direct interp={interp}")
    n, ft = 32, 64
    bm, ps = dataset(n, 10, 90, n, seed=13)
    d = ps.images.cuda()
    recs = {}
    for method in (1, 0):
        r = Reconstruction(n, n, ft, 1.5, ctf_action=1, interp=interp, method=method,
                           flags=abi.BSX_FLAG_FOM, nhalves=2)
        r.insert(d, ps.parts)
        recs[method] = r
    for half in (0, 1):
        a0, a = recs[1].accumulators(half), recs[0].accumulators(half)
        for q in range(5):
            e = ((a[q] - a0[q]).abs().max() / a0[q].abs().max()).item()
            assert e < 2e-5, (half, q, e)
    f0 = recs[1].finish(want_fom=True)
    f1 = recs[0].finish(want_fom=True)
    assert ((f1.map - f0.map).abs().max() / f0.map.abs().max()).item() < 1e-5
    assert ((f1.fom - f0.fom).abs().max() / f0.fom.abs().max()).item() < 1e-4
    for r in recs.values():
        r.close()


@pytest.mark.parametrize("interp", [0, 1, 2])
@pytest.mark.parametrize("ft,box,n,fom", [(32, 16, 16, True), (128, 61, 64, True), (128, 61, 64, False),
                                          (256, 90, 96, True), (256, 90, 96, False),
                                          (512, 200, 128, True)])
def test_specialised_fills_match_direct(ft, box, n, fom, interp):
    """The fills specialised on the interpolation, with and without the FOM
    sums, over the transform sizes and boxes that leave rows and columns
    empty: every accumulator plane matches the direct-atomic path, which
    computes the same terms, to FP32 summation order (40 particles, at most
    about 2^9 terms a voxel of random rounding: 2e-5 of the maximum)."""
    say(f"fills ft={ft} box={box} n={n} fom={fom} interp={interp}")
    bm, ps = dataset(box, 10, 40, box, seed=ft + box)
    d = ps.images.cuda()
    acc = []
    for method in (1, 0):
        r = Reconstruction(n, box, ft, 1.5, ctf_action=1, interp=interp, method=method,
                           flags=abi.BSX_FLAG_FOM if fom else 0)
        r.insert(d, ps.parts)
        acc.append(r.accumulators(0))
        r.close()
    for q, (a0, a) in enumerate(zip(*acc)):
        assert (a - a0).abs().max() <= 2e-5 * a0.abs().max(), q


@pytest.mark.parametrize("interp", [0, 1, 2])
def test_ewald_pairs_match_direct(interp):
    """With the Ewald offsets the binned insertion emits each frequency at
    +m_z and -m_z as pair entries that stand for the mate's -m_z and +m_z
    emissions: the accumulators match the direct-atomic path (method 1),
    which computes all four emissions, to FP32 summation order. 1 kV makes
    the offsets span several voxels."""
    say(f"Ewald pairs vs direct interp={interp}")
    n, ft = 32, 64
    bm, ps = dataset(n, 10, 90, n, seed=14)
    parts = ps.parts.copy()
    parts["volt"] = 1e3
    d = ps.images.cuda()
    acc = {}
    for method in (1, 0):
        r = Reconstruction(n, n, ft, 1.5, ctf_action=1, interp=interp, method=method,
                           flags=abi.BSX_FLAG_EWALD)
        r.insert(d, parts)
        acc[method] = r.accumulators(0)
        r.close()
    for q in range(3):
        e = ((acc[0][q] - acc[1][q]).abs().max() / acc[1][q].abs().max()).item()
        assert e < 2e-5, (q, e)


def test_graph_cache_of_chunked_inserts():
    """BSX_FLAG_GRAPH keeps one graph per (images, count, tuning): three
    chunks inserted after each other are each captured on their second
    appearance and replayed on the third (6 graph launches in all), an
    insert that reallocates the record buffers in between drops the cache
    instead of replaying graphs that hold the old buffers, and every pass
    gives the single-insert accumulators."""
    import ctypes as C
    from bsoft_amd.abi import call
    bm, ps = dataset(32, 10, 300, 32, seed=12)
    d = ps.images.cuda()
    ref = Reconstruction(32, 32, 64, 1.5, ctf_action=1, batch=64)
    ref.insert(d, ps.parts)
    a0 = ref.accumulators(0)
    g = Reconstruction(32, 32, 64, 1.5, ctf_action=1, batch=64, flags=abi.BSX_FLAG_GRAPH)
    bounds = [0, 90, 200, 300]

    def chunked():
        g.reset()
        for lo, hi in zip(bounds, bounds[1:]):
            g.insert(d[lo:hi], ps.parts[lo:hi])
        torch.cuda.synchronize()
        a = g.accumulators(0)
        return float((a[:3] - a0[:3]).abs().max() / a0[:3].abs().max())

    nl = C.c_int64()
    g.insert(d, ps.parts)   # sizes the record buffers for every chunk
    for rep in range(3):
        err = chunked()
        call("bsx_recon_graph_launches", g.h, C.byref(nl))
        say(f"  chunked pass {rep}: max rel err {err:.2e}, graph launches {nl.value}")
        assert err <= 2e-5
        assert nl.value == 3 * max(0, rep)
    # a larger insert reallocates the records: the cached graphs are dropped
    big = torch.cat([d, d])
    bp = np.concatenate([ps.parts, ps.parts])
    g.reset()
    g.insert(big, bp)
    for rep in range(3):
        err = chunked()
        call("bsx_recon_graph_launches", g.h, C.byref(nl))
        say(f"  after reallocation, pass {rep}: max rel err {err:.2e}, graph launches {nl.value}")
        assert err <= 2e-5
        assert nl.value == 6 + 3 * max(0, rep)


def test_graph_replay_and_autotune():
    """Inserts replayed from a captured hipGraph give the eager result (the
    replay counter proves the graph ran); the autotuner leaves the handle
    empty and the chosen batch gives the same accumulators."""
    import ctypes as C
    from bsoft_amd.abi import call
    from bsoft_amd.recon import _ptr
    bm, ps = dataset(32, 10, 300, 32, seed=10)
    d = ps.images.cuda()
    ref = Reconstruction(32, 32, 64, 1.5, ctf_action=1, batch=64)
    ref.insert(d, ps.parts)
    a0 = ref.accumulators(0)
    g = Reconstruction(32, 32, 64, 1.5, ctf_action=1, batch=64, flags=abi.BSX_FLAG_GRAPH)
    for rep in range(4):
        g.reset()
        g.insert(d, ps.parts)
        torch.cuda.synchronize()
        a = g.accumulators(0)
        assert (a[:3] - a0[:3]).abs().max() <= 2e-5 * a0[:3].abs().max(), rep
        torch.cuda.synchronize()
    nl = C.c_int64()
    call("bsx_recon_graph_launches", g.h, C.byref(nl))
    say(f"  graph replays {nl.value}")
    assert nl.value == 3            # the first insert runs eagerly, the second is captured
    t = Reconstruction(32, 32, 64, 1.5, ctf_action=1, batch=256)
    cb, ms = C.c_int32(), C.c_double()
    parts = np.ascontiguousarray(ps.parts)
    call("bsx_recon_autotune", t.h, _ptr(d), synth.particles_ctypes(parts), len(parts),
         C.byref(cb), C.byref(ms), None)
    say(f"  autotune chose batch {cb.value} ({ms.value:.3f} ms)")
    assert cb.value in (32, 64, 128, 256)
    batch, piece = t.tuning()
    say(f"  tuning: batch {batch}, piece {piece}")
    assert batch == cb.value and piece in (8192, 16384, 32768)
    assert t.accumulators(0).abs().max().item() == 0
    t.insert(d, ps.parts)
    a = t.accumulators(0)
    assert (a[:3] - a0[:3]).abs().max() <= 2e-5 * a0[:3].abs().max()
    # every piece length gives the same sums
    for pl in (8192, 32768):
        t.reset()
        t.set_tuning(piece=pl)
        t.insert(d, ps.parts)
        a = t.accumulators(0)
        assert (a[:3] - a0[:3]).abs().max() <= 2e-5 * a0[:3].abs().max(), pl


def _star_project(tmp_path):
    from bsoft_amd import formats
    bm, ps = dataset(32, 10, 60, 32, seed=11)
    n = len(ps.parts)
    formats.write_mrc(str(tmp_path / "p.mrcs"), ps.images.numpy(), (1.5, 1.5, 1.0), (16, 16, 0),
                      images=n)
    rows = [[i + 1, ps.parts["def_avg"][i], 16, 16, *ps.parts["view"][i][:3],
             math.degrees(ps.parts["view"][i][3]), 1] for i in range(n)]
    b = formats.StarBlock(name="m", items={
        "micrograph.id": "m", "micrograph.pixel_size_x": "1.5", "particle.file_name": "p.mrcs",
        "ctf.voltage": "300000", "ctf.Cs": "27000000", "ctf.amplitude_phase_shift":
        repr(float(ps.parts["amp_shift"][0])), "ctf.defocus_average": "20000"},
        loops=[(["particle.id", "particle.defocus", "particle.origin_x", "particle.origin_y",
                 "particle.view_x", "particle.view_y", "particle.view_z", "particle.view_angle",
                 "particle.select"], rows)])
    star = str(tmp_path / "proj.star")
    formats.write_star(star, [b])
    return star, ps


def _oracle_maps(ps, nmaps, **kw):
    """The FP64 oracle's maps (imap 0..nmaps-1) of the particles in project
    order with T = 2 round-robin partial maps, as breconstruct runs it."""
    d = dict(size=32, box=32, ft_size=64, interp=0, sampling=1.5, hi_res=1.5, lo_res=0.0,
             ctf_action=1, flags=0, wiener=0.0, nhalves=1, batch=0, mem_cap=0)
    d.update(kw)
    o = OracleRecon(ReconParams(**d), 2, 64)
    o.insert(synth.particles_list(ps.parts), ps.images.numpy())
    return [o.finish(i, nmaps, want_fom=bool(d["flags"] & abi.BSX_FLAG_FOM)) for i in range(nmaps)]


def test_breconstruct_cli_on_star_project(tmp_path, capsys):
    """breconstruct over a STAR project and an MRC stack, full map and half
    maps (-fullmap -halfmaps: <name>, <name>_01, <name>_02) against the FP64
    oracle on the same particles, written as MRC with the sampling and
    origin of the reference's output; the FOM maps too (-fom)."""
    from bsoft_amd import breconstruct, formats
    star, ps = _star_project(tmp_path)
    out = str(tmp_path / "map.mrc")
    fom = str(tmp_path / "fom.mrc")
    assert breconstruct.main(["-reconstruction", out, "-CTF", "flip", "-fullmap", "-halfmaps",
                              "-fom", fom, "-verbose", star]) == 0
    printed = capsys.readouterr().out
    assert "SNR(0.5):" in printed and "FSC(0.3):" in printed and "Radius\ts(1/A)" in printed
    ref = _oracle_maps(ps, 3, flags=abi.BSX_FLAG_FOM)
    for name, (m, f, _, st) in zip(("map.mrc", "map_01.mrc", "map_02.mrc"), ref):
        g = formats.read_mrc(str(tmp_path / name))
        assert g.data.shape == (1, 32, 32, 32) and g.sampling == pytest.approx((1.5,) * 3)
        assert g.origin == pytest.approx((16, 16, 16))
        err = np.abs(g.data[0] - m).max() / np.abs(m).max()
        say(f"  {name}: max rel err {err:.2e} vs the oracle")
        assert err <= 1e-4
    gf = formats.read_mrc(str(tmp_path / "fom_01.mrc")).data[0].astype(np.float64)
    of = ref[1][1]
    sel = np.abs(of) > 1e-3
    assert np.median(np.abs(gf[sel] - of[sel]) / np.abs(of[sel])) < 1e-3
    # -halfmaps alone: the two half maps only
    out2 = str(tmp_path / "h.mrc")
    assert breconstruct.main(["-reconstruction", out2, "-CTF", "1", "-halfmaps", star]) == 0
    assert not (tmp_path / "h.mrc").exists()
    ref2 = _oracle_maps(ps, 2)
    for name, (m, _, _, _) in zip(("h_01.mrc", "h_02.mrc"), ref2):
        g = formats.read_mrc(str(tmp_path / name)).data[0]
        assert np.abs(g - m).max() <= 1e-4 * np.abs(m).max()


@pytest.mark.parametrize("ctf,action,wiener", [("baseflip", 7, 0.2), ("correct", 3, 0.2),
                                               ("apply", 2, 0.0), ("apply -wiener", 2, 0.3)])
def test_breconstruct_ctf_actions(tmp_path, ctf, action, wiener):
    """-CTF spellings of include/options.h:418-442: baseflip and correct are
    Wiener filters with the default factor 0.2 (breconstruct.cpp:187),
    apply applies the CTF, and apply with -wiener is a Wiener filter."""
    from bsoft_amd import breconstruct, formats
    star, ps = _star_project(tmp_path)
    out = str(tmp_path / "c.mrc")
    args = ["-reconstruction", out, "-CTF", ctf.split()[0], star]
    if "-wiener" in ctf:
        args[-1:-1] = ["-wiener", str(wiener)]
    assert breconstruct.main(args) == 0
    (m, _, _, _), = _oracle_maps(ps, 1, ctf_action=action, wiener=wiener)
    g = formats.read_mrc(out).data[0]
    assert np.abs(g - m).max() <= 1e-4 * np.abs(m).max()


def test_breconstruct_trilinear_rescale(tmp_path):
    """-interpolate trilinear -rescale avg,std: particles normalised before
    insertion, the map rescaled to (avg, std) and then given the sinc^2
    correction of trilinear insertion (Bimage::filter_sinc), as
    breconstruct.cpp:336 and :359 do, against the oracle's chain."""
    from bsoft_amd import breconstruct, formats
    star, ps = _star_project(tmp_path)
    out = str(tmp_path / "t.mrc")
    assert breconstruct.main(["-reconstruction", out, "-CTF", "flip", "-interpolate", "trilinear",
                              "-rescale", "0.5,2", star]) == 0
    (m, _, _, _), = _oracle_maps(ps, 1, interp=2, flags=abi.BSX_FLAG_RESCALE)
    o = Oracle(64)
    m = o.filter_sinc(o.rescale_to_avg_std(m, 0.5, 2.0), (16, 16, 16))
    g = formats.read_mrc(out).data[0].astype(np.float64)
    err = np.abs(g - m).max() / np.abs(m).max()
    say(f"  trilinear + rescale + sinc: max rel err {err:.2e}")
    assert err <= 1e-4


@pytest.mark.parametrize("mode", [1, 2])
def test_breconstruct_symmetry_modes(tmp_path, mode):
    """-mode 1: the particles inserted once, then the map symmetrized in real
    space (the FP64 restatement of Bimage::symmetrize on the direct API's
    map); -mode 2: each particle inserted once at the related view that
    random_symmetric_views draws with the same seed."""
    from bsoft_amd import breconstruct, formats
    from bsoft_amd.recon import random_symmetric_views
    from oracle import sym_ref
    say(f"breconstruct -mode {mode}")
    star, ps = _star_project(tmp_path)
    out = str(tmp_path / "map.mrc")
    assert breconstruct.main(["-reconstruction", out, "-CTF", "flip", "-symmetry", "C3",
                              "-mode", str(mode), "-seed", "5", star]) == 0
    got = formats.read_mrc(out).data[0]
    rec = Reconstruction(32, 32, 64, 1.5, ctf_action=1)
    parts = ps.parts.copy()
    if mode == 2:
        parts["view"] = random_symmetric_views("C3", parts["view"], np.random.default_rng(5))
    rec.insert(ps.images.cuda().contiguous(), parts)
    ref = rec.finish(0, 1).map.cpu().numpy()
    if mode == 1:
        ref = sym_ref.symmetrize(ref, "C3", (16, 16, 16))
    assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("sym", ["C3", "D2", "O"])
def test_symmetry_equals_expanded_particles(sym):
    """Point-group symmetry (fspace_pack_2D over symmetry_get_all_views) adds
    each particle at all its related views: the same sums as inserting the
    explicitly expanded particle list, up to FP32 summation order; the
    particle count stays that of the input."""
    say(f"symmetry {sym}")
    n = 12
    bm, ps = dataset(64, 10, n, 64, seed=12)
    d = ps.images.cuda()
    r = Reconstruction(64, 64, 128, 1.5, ctf_action=1)
    r.set_symmetry(sym)
    r.insert(d, ps.parts)
    sv = symmetry_views(sym, ps.parts["view"])
    order = sv.shape[1]
    ex = np.repeat(ps.parts, order)
    ex["view"] = sv.reshape(-1, 4)
    r2 = Reconstruction(64, 64, 128, 1.5, ctf_action=1)
    r2.insert(d.repeat_interleave(order, dim=0).contiguous(), ex)
    a, b = r.accumulators(0), r2.accumulators(0)
    for q in range(3):
        e = ((a[q] - b[q]).abs().max() / b[q].abs().max()).item()
        assert e < 2e-5, (sym, q, e)
    g = r.finish()
    assert g.particles == n
    assert g.weight_sum == pytest.approx(r2.finish().weight_sum, rel=1e-6)


@pytest.mark.parametrize("interp,tilted", [(0, False), (1, False), (2, False), (0, True)])
def test_two_d_reconstruction(interp, tilted):
    """breconstruct -TwoD (BSX_FLAG_2D): one z plane, z real size 1 in the
    coordinates and the taper. Views along +z or -z with in-plane angles (the
    class-average use), or tilted 3D views with nearest-neighbour insertion
    (their trilinear corners leave the reference's single plane through its
    one-step wrap, which is undefined there). The map, transform, coverage
    and Friedel residual against the FP64 oracle."""
    from types import SimpleNamespace
    bm, ps = dataset(32, 10, 200, 32, seed=13)
    parts = ps.parts.copy()
    if not tilted:
        rng = np.random.default_rng(13)
        sgn = np.where(rng.random(len(parts)) < 0.5, -1.0, 1.0)
        ang = parts["view"][:, 3]
        parts["view"] = np.stack([0 * ang, 0 * ang, sgn, ang], axis=1)
    rec, g, ref, o = run_pair(SimpleNamespace(parts=parts, images=ps.images), size=32, box=32,
                              ft=64, interp=interp, flags=abi.BSX_FLAG_2D)
    m, _, ftc, st = ref
    assert g.map.shape == (1, 32, 32) and m.shape == (1, 32, 32)
    if interp == 0 and not tilted:     # the command line gives the same plane
        from bsoft_amd import breconstruct, formats
        import tempfile
        with tempfile.TemporaryDirectory() as d:
            import pathlib
            star, ps2 = _star_project(pathlib.Path(d))
            out = str(pathlib.Path(d) / "map2d.mrc")
            assert breconstruct.main(["-reconstruction", out, "-TwoD", star]) == 0
            mm = formats.read_mrc(out)
            assert mm.data.shape == (1, 1, 32, 32)
            assert mm.origin == pytest.approx((16, 16, 0))
    gm = g.map.cpu().numpy().astype(np.float64)
    err = np.abs(gm - m).max() / np.abs(m).max()
    fe = np.abs(g.ft.cpu().numpy() - ftc).max() / np.abs(ftc).max()
    say(f"  2D max rel err map {err:.3e} transform {fe:.3e} coverage {g.coverage}/{st.coverage}")
    assert err <= 1e-4 and fe <= 1e-4
    assert g.coverage == st.coverage and g.particles == st.particles
    assert abs(g.friedel - st.friedel) <= 1e-3 * st.friedel + 1e-5 * np.abs(ftc).max()


@pytest.mark.parametrize("first", [False, True])
def test_reset_recorded_in_a_graph(first):
    """A reset recorded into a graph clears what inserts leave, whether the
    handle was empty or not when it was recorded, and on every replay, with the
    program's own inserts, resets and finishes in between."""
    rng = np.random.default_rng(3)
    ps = synth.make_particles(synth.make_blob_map(32, 8, rng), 40, 32, rng, seed=3)
    imgs = ps.images.cuda().contiguous()
    r, ref = (Reconstruction(32, 32, 64, 1.5, ctf_action=1) for _ in range(2))
    ref.insert(imgs, ps.parts)
    want = ref.finish().map
    say(f"recorded reset, inserts before: {first}")
    if first:
        r.insert(imgs, ps.parts)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        r.reset()
    for _ in range(3):
        r.insert(imgs, ps.parts)
        g.replay()
        r.insert(imgs, ps.parts)
        assert (r.finish().map - want).abs().max() <= 1e-5 * want.abs().max()
        torch.cuda.synchronize()
        r.reset()
        r.insert(imgs, ps.parts)
        assert (r.finish().map - want).abs().max() <= 1e-5 * want.abs().max()


def test_accumulators_recorded_in_a_graph():
    """Reading the sums (bsx_recon_accumulators, no allocation), recorded while
    the handle was empty, gives the sums of the inserts before each replay."""
    rng = np.random.default_rng(4)
    ps = synth.make_particles(synth.make_blob_map(32, 8, rng), 40, 32, rng, seed=4)
    imgs = ps.images.cuda().contiguous()
    r, ref = (Reconstruction(32, 32, 64, 1.5, ctf_action=1) for _ in range(2))
    planes = torch.zeros((5, 32, 32, 32), device="cuda")
    say("recorded accumulators")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        abi.call("bsx_recon_accumulators", r.h, 0, planes.data_ptr(), torch.cuda.current_stream().cuda_stream)
    for half in (imgs[:25], imgs[25:]):
        part = ps.parts[:25] if len(half) == 25 else ps.parts[25:]
        r.insert(half.contiguous(), part)
        ref.insert(half.contiguous(), part)
        g.replay()
        torch.cuda.synchronize()
        want = ref.accumulators(0)
        for a, b in zip(planes[:3], want[:3]):
            assert (a - b).abs().max() <= 1e-5 * b.abs().max()
    assert (r.finish().map - ref.finish().map).abs().max() <= 1e-5 * ref.finish().map.abs().max()


@pytest.mark.parametrize("size,flags,interp", [(32, 0, 0), (24, abi.BSX_FLAG_FOM, 0), (32, abi.BSX_FLAG_2D, 1),
                                               (48, 0, 2)])
def test_finish_insert_and_reset_in_any_order(size, flags, interp):
    """The finish folds the binned sums and clears them, a later insert adds to
    the folded ones, and a reset clears what an unfinished insert left: the
    maps of each half and their coverage equal those of a fresh handle given
    the same particles (FP32 summation order: 1e-5 of the maximum)."""
    rng = np.random.default_rng(size)
    ps = synth.make_particles(synth.make_blob_map(size, 8, rng), 60, size, rng, seed=size)
    if flags & abi.BSX_FLAG_2D:
        ps.parts["view"] = [0, 0, 1, 0.3]
    imgs = ps.images.cuda().contiguous()
    fom = bool(flags & abi.BSX_FLAG_FOM)

    def fresh():
        return Reconstruction(size, size, part_ft_size(size, 1, 2), 1.5, ctf_action=1, flags=flags,
                              interp=interp, nhalves=2)

    def outputs(r):
        return [r.finish(i, 3, want_fom=fom) for i in range(3)]

    def same(a, b):
        for x, y in zip(a, b):
            assert x.coverage == y.coverage and x.particles == y.particles
            assert x.weight_sum == pytest.approx(y.weight_sum, rel=1e-6)
            assert (x.map - y.map).abs().max() <= 1e-5 * y.map.abs().max()
            if fom:
                assert torch.allclose(x.fom, y.fom, rtol=1e-3, atol=1e-3)

    r = fresh()
    say(f"finish order size={size} ft={r.params.ft_size} flags={flags} interp={interp}")
    r.insert(imgs[:20], ps.parts[:20])
    outputs(r)
    r.insert(imgs[20:50].contiguous(), ps.parts[20:50])
    both = outputs(r)
    ref = fresh()
    ref.insert(imgs[:50].contiguous(), ps.parts[:50])
    same(both, outputs(ref))
    r.insert(imgs[50:].contiguous(), ps.parts[50:])
    r.reset()
    r.insert(imgs[:20], ps.parts[:20])
    ref.reset()
    ref.insert(imgs[:20], ps.parts[:20])
    same(outputs(r), outputs(ref))
