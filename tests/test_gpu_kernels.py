"""GPU parity of the FFT, map transform, extraction, FSC and FRC kernels
against the FP64 CPU oracle / the textbook DFT, through the C-ABI."""
import math
import sys

import numpy as np
import pytest
import torch

from bsoft_amd import bresolve, recon, synth
from oracle import resolution_ref
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("shape,dims", [((16,), 1), ((512,), 1), ((24,), 1), ((384,), 1),
                                        ((7, 128), 1), ((3, 64, 256), 2), ((2, 512, 512), 2),
                                        ((96, 32), 2), ((4, 192, 96), 2), ((32, 32, 32), 3),
                                        ((64, 64, 64), 3), ((2, 48, 48, 48), 3),
                                        ((128, 256, 64), 3)])
@pytest.mark.parametrize("direction", [-1, 1])
def test_fft_vs_textbook(gpu, shape, dims, direction):
    say(f"fft shape={shape} dims={dims} dir={direction}")
    rng = np.random.default_rng(sum(shape))
    x = (rng.normal(size=shape) + 1j * rng.normal(size=shape)).astype(np.complex64)
    t = torch.from_numpy(x).cuda()
    recon.fft(t, dims, direction, norm=1)
    axes = tuple(range(len(shape) - dims, len(shape)))
    xd = x.astype(np.complex128)
    n = int(np.prod([shape[a] for a in axes]))
    ref = np.fft.fftn(xd, axes=axes) if direction < 0 else np.fft.ifftn(xd, axes=axes) * n
    ref /= math.sqrt(n)
    err = np.abs(t.cpu().numpy() - ref).max() / np.abs(ref).max()
    say(f"  rel err {err:.2e}")
    assert err < 2e-6


def test_map_transform_vs_oracle(gpu):
    rng = np.random.default_rng(1)
    bm = synth.make_blob_map(64, 20, rng)
    vol = bm.volume()
    ft = recon.map_transform(vol.cuda(), (32, 32, 32))
    ref = Oracle(64).map_transform(vol.numpy().astype(np.float64), (32, 32, 32))
    err = np.abs(ft.cpu().numpy() - ref).max() / np.abs(ref).max()
    assert err < 2e-6


@pytest.mark.parametrize("kw,kp", [(8, 2), (10, 2), (4, 1)])
def test_extract_vs_oracle(gpu, kw, kp):
    rng = np.random.default_rng(2)
    n = 64
    bm = synth.make_blob_map(n, 20, rng)
    vol = bm.volume()
    o = Oracle(64)
    ft_ref = o.map_transform(vol.numpy().astype(np.float64), (32, 32, 32))
    ft = torch.from_numpy(ft_ref.astype(np.complex64)).cuda()
    views = np.vstack([synth.uniform_views(12, rng), [[0, 0, 1, 0], [0, 0, 1, math.pi / 2]]])
    mats = synth.view_to_matrix(views)
    secs = recon.central_sections(ft, mats, 1.5, 3.0, kw, kp, center=True).cpu().numpy()
    for i, m in enumerate(mats):
        ref = o.central_section(ft_ref, 1.5, m, 3.0, kw, kp, 1)
        err = np.abs(secs[i] - ref).max() / np.abs(ref).max()
        assert err < 1e-5, (i, err)


def test_fsc_vs_oracle(gpu):
    rng = np.random.default_rng(3)
    n = 48
    a = (rng.normal(size=(n, n, n)) + 1j * rng.normal(size=(n, n, n))).astype(np.complex64)
    b = (a + 0.7 * (rng.normal(size=(n, n, n)) + 1j * rng.normal(size=(n, n, n)))).astype(np.complex64)
    f = recon.fsc(torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda(), 1.5, 1.5)
    ref = Oracle(64).fsc(a, b, 1.5, 1.5)
    assert len(f) == len(ref)
    np.testing.assert_allclose(f, ref, atol=1e-9)


def test_frc_score_vs_oracle(gpu):
    rng = np.random.default_rng(4)
    n = 64
    P = (rng.normal(size=(5, n, n)) + 1j * rng.normal(size=(5, n, n))).astype(np.complex64)
    R = (P[[1, 0, 3, 2, 4]] + 0.5 * (rng.normal(size=(5, n, n)) + 1j * rng.normal(size=(5, n, n)))).astype(np.complex64)
    pairs = np.array([[i, j] for i in range(5) for j in range(5)], np.int32)
    s = recon.img_recip_space_fom(torch.from_numpy(P).cuda(), torch.from_numpy(R).cuda(), pairs, 1.5, 4.0, 50.0)
    o = Oracle(64)
    ref = [o.recip_space_fom(P[i], R[j], 1.5, 4.0, 50.0)[0] for i, j in pairs]
    np.testing.assert_allclose(s, ref, atol=1e-9)
    with pytest.raises(Exception):
        recon.img_recip_space_fom(torch.from_numpy(P).cuda(), torch.from_numpy(R).cuda(),
                                  np.array([[0, 5]], np.int32), 1.5, 4.0)


@pytest.mark.parametrize("shape,dims", [((3, 24, 96), 2), ((5, 48, 24), 2), ((1, 384, 16), 2), ((24, 48, 96), 3),
                                        ((16, 16, 16), 3), ((2, 192, 24, 16), 3), ((512, 16, 16), 3)])
def test_fft_ragged_line_bundles(shape, dims):
    """Axis transforms whose numbers of lines are no multiple of a workgroup's
    bundle, against numpy's FP64 transform (2e-6 of the maximum, FP32 rounding
    over at most 27 butterfly stages)."""
    rng = np.random.default_rng(sum(shape))
    x = (rng.normal(size=shape) + 1j * rng.normal(size=shape)).astype(np.complex64)
    say(f"fft shape={shape} dims={dims}")
    axes = tuple(range(len(shape) - dims, len(shape)))
    ref = np.fft.fftn(x.astype(np.complex128), axes=axes, norm="ortho")
    got = recon.fft(torch.as_tensor(x).cuda(), dims, -1, 1).cpu().numpy()
    assert np.abs(got - ref).max() <= 2e-6 * np.abs(ref).max()


@pytest.mark.parametrize("n,origin", [(16, (8, 8, 8)), (24, (11.5, 12, 3.25)), (48, (0, 24, 47)), (96, (48, 48, 48))])
def test_map_transform_origin(n, origin):
    """Map transform of a real map moved to an origin that is no grid centre,
    against numpy (1e-6 of the maximum)."""
    rng = np.random.default_rng(n)
    v = rng.normal(size=(n, n, n)).astype(np.float32)
    say(f"map transform n={n} origin={origin}")
    f = np.fft.fftfreq(n, 1 / n)
    ph = 2j * np.pi / n * (f[None, None, :] * origin[0] + f[None, :, None] * origin[1] + f[:, None, None] * origin[2])
    ref = np.fft.fftn(v.astype(np.float64), norm="ortho") * np.exp(ph)
    got = recon.map_transform(torch.as_tensor(v).cuda(), origin).cpu().numpy()
    assert np.abs(got - ref).max() <= 1e-6 * np.abs(ref).max()


@pytest.mark.parametrize("shape", [(16, 16, 16), (24, 24, 24), (96, 96), (1, 48, 48)])
def test_fsc_dpr_with_empty_transforms(shape):
    """FSC and DPR where one map has no power, or both have none: the shells'
    phase difference is then the other value's angle, weighed with its power."""
    rng = np.random.default_rng(len(shape))
    v = torch.as_tensor(rng.normal(size=shape).astype(np.float32)).cuda()
    z = torch.zeros_like(v)
    say(f"fsc_dpr shape={shape}")
    s, fsc, dpr = bresolve.fsc_dpr(z, z, 1.5)
    assert np.all(fsc[1:] == 0) and np.all(dpr == 0)
    s, fsc, dpr = bresolve.fsc_dpr(v, z, 1.5)
    ref = resolution_ref.fsc_dpr(v.cpu().numpy().astype(np.float64), np.zeros(shape), 1.5)
    np.testing.assert_allclose(fsc, ref[1], atol=1e-6)
    np.testing.assert_allclose(dpr, ref[2], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("n,width", [(24, 3), (24, 8), (32, 5), (48, 4), (48, 9), (96, 10), (64, 7), (20, 6), (21, 8)])
def test_sections_of_every_tile_path(n, width):
    """Central sections against the FP64 oracle for kernel widths on both sides
    of the LDS box rule, edges that are no multiple of the 8 x 8 tile, views
    along the axes, and a matrix that shrinks the plane (its box has repeated
    taps); FP32 rounding: 1e-5 of the maximum."""
    rng = np.random.default_rng(n + width)
    ft = (rng.normal(size=(n, n, n)) + 1j * rng.normal(size=(n, n, n))).astype(np.complex64)
    mats = np.concatenate([np.eye(3)[None], synth.view_to_matrix([[1, 0, 0, 0.3], [0, 0, -1, 1.0]]),
                           synth.view_to_matrix(synth.uniform_views(4, rng)), 0.3 * np.eye(3)[None]])
    say(f"sections n={n} width={width} views={len(mats)}")
    out = recon.central_sections(torch.as_tensor(ft).cuda(), mats, 1.5, 1.5, width, 2, True).cpu().numpy()
    o = Oracle(64)
    for i, m in enumerate(mats):
        ref = o.central_section(ft, 1.5, m, 1.5, width, 2, 1)
        assert np.abs(out[i] - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("n,width", [(24, 5), (40, 6), (33, 7), (48, 8), (64, 9), (96, 10), (2, 8), (3, 5), (10, 10)])
def test_sections_of_boxes_beyond_lds(n, width):
    """Sections whose taps do not fit an LDS box (matrices that stretch the
    plane; maps smaller than the kernel, with several periodic wraps) are
    shared among a tile's wavefronts like the others: against the FP64 oracle,
    FP32 rounding (1e-5 of the maximum)."""
    rng = np.random.default_rng(n + width)
    ft = (rng.normal(size=(n, n, n)) + 1j * rng.normal(size=(n, n, n))).astype(np.complex64)
    mats = np.array([[[1, 1, 0], [1, -1, 0], [1, 1, 0]], [[1, -1, 1], [-1, 1, 1], [1, 1, 1]],
                     [[0, 1, 0], [1, 0, 0], [0, 0, 1]]], dtype=float)
    say(f"sections beyond LDS n={n} width={width}")
    out = recon.central_sections(torch.as_tensor(ft).cuda(), mats, 1.5, 1.5, width, 2, True).cpu().numpy()
    o = Oracle(64)
    for i, m in enumerate(mats):
        ref = o.central_section(ft, 1.5, m, 1.5, width, 2, 1)
        assert np.abs(out[i] - ref).max() <= 1e-5 * np.abs(ref).max()


def test_sections_beyond_lds_take_no_longer_than_their_taps():
    """Sections of matrices that stretch the plane, whose taps come from memory,
    take at most eight times as long as those of rotations at width 10 (12
    times with one of a tile's wavefronts at work)."""
    ft = torch.randn((128, 128, 128), dtype=torch.complex64, device="cuda")
    wide = np.tile(np.array([[1, 1, 0], [1, -1, 0], [1, 1, 0]], dtype=float), (200, 1, 1))
    rot = synth.view_to_matrix(synth.uniform_views(200, np.random.default_rng(1)))

    def best(mats):
        took = []
        for _ in range(6):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            recon.central_sections(ft, mats, 1.5, 3.0, 10, 2)
            b.record()
            b.synchronize()
            took.append(a.elapsed_time(b))
        return min(took[1:])

    say("sections beyond LDS, time")
    w, r = best(wide), best(rot)
    say(f"  {w:.3f} ms against {r:.3f} ms")
    assert w <= 8 * r


@pytest.mark.parametrize("n,width,views", [(256, 8, 16385), (24, 3, 65535)])
def test_sections_of_very_many_views(n, width, views):
    """More sections than one launch has threads for (2^32 threads from 16,385
    sections of 256^2 on), and the most views that are accepted: sections at both
    ends and on both sides of every launch equal those of a call of their own."""
    rng = np.random.default_rng(views)
    ft = torch.randn((n, n, n), dtype=torch.complex64, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    some = synth.view_to_matrix(synth.uniform_views(7, rng))
    pick = np.arange(views) % 7
    say(f"sections n={n} width={width} views={views}")
    out = recon.central_sections(ft, some[pick], 1.5, 3.0, width, 2, True)
    want = recon.central_sections(ft, some, 1.5, 3.0, width, 2, True)
    for v in (0, 1, views // 2 - 1, views // 2, 8191, 8192, 16383, views - 2, views - 1):
        assert torch.equal(torch.view_as_real(out[v]), torch.view_as_real(want[pick[v]])), v


def test_workspaces_given_back():
    """release_workspaces frees what earlier calls kept, so that other users of
    the device get it; the calls after it give the same values."""
    rng = np.random.default_rng(5)
    v = [torch.as_tensor(rng.normal(size=(192, 192, 192)).astype(np.float32)).cuda() for _ in range(2)]
    say("workspaces given back")
    one = bresolve.fsc_dpr(*v, 1.5)
    torch.cuda.synchronize()
    kept = torch.cuda.mem_get_info()[0]
    recon.release_workspaces()
    # the two half transforms of the call
    assert torch.cuda.mem_get_info()[0] - kept >= 2 * 96 * 192 * 192 * 8
    for a, b in zip(one, bresolve.fsc_dpr(*v, 1.5)):
        np.testing.assert_allclose(a, b, rtol=1e-9, atol=1e-12)


def test_workspaces_shared_by_threads_and_streams():
    """Calls without a handle keep their workspaces between calls: four threads,
    each on a stream of its own and with sizes of its own, get the results of
    the same calls made one after the other."""
    import threading
    rng = np.random.default_rng(8)
    work = []
    for n in (32, 48, 64, 32):
        a = torch.as_tensor(rng.normal(size=(n, n, n)).astype(np.float32)).cuda()
        b = torch.as_tensor(rng.normal(size=(n, n, n)).astype(np.float32)).cuda()
        work.append((a, b, synth.uniform_views(5, rng)))

    def one(a, b, views):
        s, fsc, dpr = bresolve.fsc_dpr(a, b, 1.5)
        ft = recon.map_transform(a)
        return fsc, dpr, recon.project(ft, views, 1.5, 3.0, 5).cpu().numpy()

    want = [one(*w) for w in work]
    torch.cuda.synchronize()
    bad = []

    def loop(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(10):
                got = one(*work[i])
                for g, w in zip(got, want[i]):
                    if not np.allclose(g, w, rtol=1e-9, atol=1e-12):
                        bad.append(i)

    say("workspaces: 4 threads x 10 rounds")
    ts = [threading.Thread(target=loop, args=(i,)) for i in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
