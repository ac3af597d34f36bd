"""Symmetric geometries, where one ray coordinate serves several pixels or rays: against the
FP64 oracle at the edges of the form (odd and even sides, bins and angles, tiles and
windows that end inside the image, the grids that only one of the symmetries fits)."""
import ctypes
import math

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

REL = 1e-5  # the FP32 operators' bar against the oracle
PI = math.pi

# (n, R, A, sinogram corners): [0, pi) on the default grid has both symmetries, [0, 2 pi) and
# a limited arc only the half turn, a shifted detector none
GEO = [
    (2, 2, 1, (0.0, 1.0, PI, -1.0)), (3, 2, 2, (0.0, 1.0, PI, -1.0)), (5, 7, 3, (0.0, 1.0, PI, -1.0)),
    (31, 33, 8, (0.0, 1.0, PI, -1.0)), (32, 64, 9, (0.0, 1.0, PI, -1.0)), (33, 31, 16, (0.0, 1.0, PI, -1.0)),
    (63, 65, 17, (0.0, 1.42, PI, -1.42)), (64, 63, 40, (0.0, 0.7, PI, -0.7)), (65, 128, 41, (0.0, 1.0, PI, -1.0)),
    (97, 97, 66, (0.0, 1.0, PI, -1.0)), (130, 131, 47, (0.0, 1.0, PI, -1.0)), (96, 160, 65, (0.0, 1.0, 2 * PI, -1.0)),
    (65, 65, 20, (0.0, 1.0, 2.0, -1.0)), (66, 90, 34, (0.1, 1.0, PI + 0.1, -1.0)), (67, 67, 33, (0.0, 1.03, PI, -0.97)),
]


def _rel(a, b):
    return np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-300)


def _geo(sc):
    return dict(sino_tl=(sc[0], sc[1]), sino_br=(sc[2], sc[3]))


@pytest.mark.parametrize("n,R,A,sc", GEO)
def test_backprojection_planes(n, R, A, sc):
    import torch
    from pyraft_amd.device import BP_NVARIANTS, Plan
    s = np.random.default_rng(n + R + A).random((3, R, A)).astype(np.float32)
    ref = np.stack([O.backprojection(v.astype(np.float64), n, **_geo(sc)) for v in s])
    j0, j1 = A // 3, max(A // 3 + 1, A - 1)
    part = np.zeros_like(s, dtype=np.float64)
    part[:, :, j0:j1] = s[:, :, j0:j1]
    pref = np.stack([O.backprojection(v, n, **_geo(sc)) for v in part])
    x = torch.from_numpy(s).cuda()
    for v in range(BP_NVARIANTS):
        p = Plan(n, R, A, sino_corners=sc)
        p.set_bp_variant(v)
        print("planes", n, R, A, sc, "variant", v, flush=True)
        assert _rel(p.backprojection(x).cpu().numpy(), ref) <= REL
        assert _rel(p.backprojection(x[1]).cpu().numpy(), ref[1]) <= REL
        assert _rel(p.backprojection(x, angles=(j0, j1)).cpu().numpy(), pref) <= REL


def _radon_close(got, ref):
    return _rel(got, ref) <= REL


@pytest.mark.parametrize("n,R,A,sc", GEO)
def test_radon_planes(n, R, A, sc):
    """Every slice count that a group of planes can end on, whole and partial ranges, and
    enough slices that the launch takes the planes undivided."""
    import torch
    from pyraft_amd.device import Plan
    p = Plan(n, R, A, sino_corners=sc)
    blocks = ((R + 127) // 128) * ((A // 2 + 8) // 8)
    many = min(-(-1024 // blocks), 1200) * 4 + 1  # odd, past SS_RADON_SLAB_BLOCKS in every form
    x = np.random.default_rng(n * A + R).random((7, n, n)).astype(np.float32)
    ref = np.stack([O.radon(v.astype(np.float64), R, A, **_geo(sc)) for v in x])
    xs = torch.from_numpy(x).cuda()
    j0, j1 = A // 3, max(A // 3 + 1, A - 1)
    for s in (1, 2, 3, 5, many):
        print("radon planes", n, R, A, sc, "slices", s, flush=True)
        idx = torch.arange(s, device="cuda") % 7
        own = ref[np.arange(s) % 7]
        got = p.radon(xs[idx]).cpu().numpy()
        assert _radon_close(got, own), s
        assert _radon_close(got[-1], own[-1]), s
        part = p.radon(xs[idx], angle_major=True, angles=(j0, j1)).cpu().numpy()
        assert _radon_close(part[:, j0:j1], own.transpose(0, 2, 1)[:, j0:j1]), s


@pytest.mark.parametrize("n,R,A,slices", [(33, 40, 9, 5), (64, 63, 17, 4), (65, 66, 24, 1201)])
def test_mesh_radon_planes(n, R, A, slices):
    import torch
    from pyraft_amd.device import Plan
    r = np.random.default_rng(n)
    t, th = np.sort(r.uniform(-1.0, 1.0, R)), np.sort(r.uniform(0.0, PI, A))
    x = r.random((4, n, n)).astype(np.float32)
    ref = np.stack([O.radon_withmesh(v.astype(np.float64), t, th) for v in x])
    p = Plan.mesh(n, t, th)
    idx = np.arange(slices) % 4
    got = p.radon(torch.from_numpy(x).cuda()[torch.from_numpy(idx).cuda()]).cpu().numpy()
    assert _rel(got, ref[idx]) <= REL and _rel(got[-1], ref[idx[-1]]) <= REL


@pytest.mark.parametrize("n,R,A,sc", GEO)
def test_transpose_planes(n, R, A, sc):
    """Both layouts, whole and partial ranges, every tile variant, and slice counts on both
    sides of the one-slice summation order."""
    import torch
    from pyraft_amd.device import Plan
    y = np.random.default_rng(3 * n + R).random((3, R, A)).astype(np.float32)
    ref = np.stack([O.radon_transpose(v.astype(np.float64), n, **_geo(sc)) for v in y])
    j0, j1 = A // 3, max(A // 3 + 1, A - 1)
    part = np.zeros_like(y, dtype=np.float64)
    part[:, :, j0:j1] = y[:, :, j0:j1]
    pref = np.stack([O.radon_transpose(v, n, **_geo(sc)) for v in part])
    p = Plan(n, R, A, sino_corners=sc)
    ys = torch.from_numpy(y).cuda()
    for s in (1, 2, 3, 11):
        print("transpose planes", n, R, A, sc, "slices", s, flush=True)
        idx = torch.arange(s, device="cuda") % 3
        own, pown = ref[np.arange(s) % 3], pref[np.arange(s) % 3]
        got = p.radon_transpose(ys[idx]).cpu().numpy()
        assert _rel(got, own) <= REL and _rel(got[-1], own[-1]) <= REL, s
        am = ys[idx].transpose(-1, -2).contiguous()
        assert np.array_equal(p.radon_transpose(am, angle_major=True).cpu().numpy(), got), s
        if np.linalg.norm(pref) > 0:
            assert _rel(p.radon_transpose(ys[idx], angles=(j0, j1)).cpu().numpy(), pown) <= REL, s
    v, times = p.tune_transpose(1, reps=1, force=True)
    assert v == -1 or _rel(p.radon_transpose(ys[0]).cpu().numpy(), ref[0]) <= REL


# (image shape, R, A, image corners, sinogram corners, slices): both symmetries, the half turn
# alone, none (stacks of slices; one or two slices take the one-ray kernels), rectangular
# images, detectors narrower and wider than the image
IC = (-1.0, 1.0, 1.0, -1.0)
LINE_GEO = [
    ((2, 2), 2, 2, IC, (0.0, 1.0, PI, -1.0), 1), ((5, 5), 7, 4, IC, (0.0, 1.0, PI, -1.0), 3),
    ((31, 31), 33, 9, IC, (0.0, 1.0, PI, -1.0), 1), ((32, 32), 64, 17, IC, (0.0, 1.0, PI, -1.0), 2),
    ((33, 33), 31, 16, IC, (0.0, 1.0, PI, -1.0), 1), ((64, 64), 63, 65, IC, (0.0, 0.7, PI, -0.7), 5),
    ((65, 65), 80, 40, IC, (0.0, 1.42, PI, -1.42), 1), ((97, 97), 97, 129, IC, (0.0, 1.0, PI, -1.0), 1),
    ((130, 130), 131, 48, IC, (0.0, 1.0, PI, -1.0), 1), ((66, 66), 90, 35, IC, (0.1, 1.0, 2.9, -1.0), 4),
    ((67, 67), 65, 33, IC, (0.0, 1.0, PI / 2 - 0.1, -1.0), 2), ((67, 67), 65, 33, IC, (0.0, 1.0, PI / 2 - 0.1, -1.0), 1),
    ((64, 64), 64, 30, IC, (0.0, 1.03, PI, -0.97), 6), ((65, 65), 65, 30, IC, (0.0, 1.03, PI, -0.97), 3),
    ((64, 64), 70, 30, IC, (0.0, 1.03, PI, -0.97), 1), ((41, 81), 90, 50, (-1.0, 0.5, 1.0, -0.5), (0.0, 1.1, PI, -1.1), 3),
    ((96, 50), 100, 41, (-0.49, 0.95, 0.49, -0.95), (0.0, 1.1, PI, -1.1), 1), ((160, 160), 41, 37, IC, (0.0, 0.2, PI, -0.2), 1),
]


def _line_matrix(shape, R, A, ic, sc):
    """(ray, pixel, length) of the line traversal as the plan defines it, traced on the host"""
    from pyraft_amd.raftypes import libraft
    d4 = ctypes.c_double * 4
    cap = 2 * sum(shape) + 8
    ij, ln = np.zeros((cap, 2), np.int32), np.zeros(cap)
    ray, pix, val = [], [], []
    for a in range(A):
        for r in range(R):
            k = libraft.raft_dda_host_ray(shape[0], shape[1], R, A, d4(*ic), d4(*sc), a, r,
                                          ij.ctypes.data_as(ctypes.POINTER(ctypes.c_int)),
                                          ln.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), cap)
            assert 0 <= k <= cap
            ray.append(np.full(k, r * A + a))
            pix.append(ij[:k, 0] * shape[1] + ij[:k, 1])
            val.append(ln[:k].copy())
    return np.concatenate(ray), np.concatenate(pix), np.concatenate(val)


@pytest.mark.parametrize("shape,R,A,ic,sc,S", LINE_GEO)
def test_line_planes(shape, R, A, ic, sc, S):
    import torch
    from pyraft_amd.device import DdaPlan
    print("line", shape, R, A, sc, S, flush=True)
    ray, pix, val = _line_matrix(shape, R, A, ic, sc)
    rng = np.random.default_rng(R + A)
    s = rng.random((S, R, A)).astype(np.float32)
    p = DdaPlan(shape, R, A, ic, sc)
    x = torch.from_numpy(s).cuda()
    t, b = p.radon_transpose(x).cpu().numpy(), p.backprojection(x).cpu().numpy()
    npix = shape[0] * shape[1]
    f = rng.random((S,) + shape).astype(np.float32)
    g = p.radon(torch.from_numpy(f).cuda()).cpu().numpy()
    for i in range(S):
        assert _rel(g[i].ravel(), np.bincount(ray, val * f[i].ravel().astype(np.float64)[pix], R * A)) <= REL
    w = np.bincount(pix, val, npix).reshape(shape)
    ok = w > 1e-6 * w.max()
    for i in range(S):
        ref = np.bincount(pix, val * s[i].ravel().astype(np.float64)[ray], npix).reshape(shape)
        assert _rel(t[i], ref) <= REL
        assert _rel(b[i][ok], ref[ok] / w[ok]) <= REL


@pytest.mark.parametrize("n,R,A,sc,S", [(2, 3, 1, (0.0, 1.0, PI, -1.0), 1), (31, 33, 7, (0.0, 1.0, PI, -1.0), 3),
                                        (33, 31, 70, (0.0, 1.0, 2 * PI, -1.0), 1), (64, 65, 150, (0.0, 0.6, PI, -0.6), 2),
                                        (65, 64, 24, (0.0, 1.03, PI, -0.97), 24), (97, 150, 66, (0.0, 1.42, 2.0, -1.42), 5)])
def test_osem_weights(n, R, A, sc, S):
    """One pass of the subsets: the update by the weights against the same steps made with the
    projectors, two slices."""
    import torch
    from pyraft_amd.device import Plan
    print("osem weights", n, R, A, sc, S, flush=True)
    rng = np.random.default_rng(n + R + A)
    y = torch.from_numpy((5 + rng.random((2, R, A))).astype(np.float32)).cuda()
    p = Plan(n, R, A, sino_corners=sc)
    got = p.em(y, 1, S).cpu().numpy()
    x = np.ones((2, n, n))
    for b in range(S):
        j0, j1 = b * A // S, (b + 1) * A // S
        on = np.zeros((R, A))
        on[:, j0:j1] = 1.0
        w = O.backprojection(on, n, **_geo(sc))
        for i in range(2):
            f = O.radon(x[i], R, A, **_geo(sc))
            rho = np.where((f > 0) & (on > 0), y[i].cpu().numpy() / np.where(f > 0, f, 1.0), 0.0)
            bp = O.backprojection(rho, n, **_geo(sc))
            x[i] = np.where(w > 0, x[i] * bp / np.where(w > 0, w, 1.0), x[i])
    assert _rel(got, x) <= REL


@pytest.mark.parametrize("n,A,S", [(2048, 60, 1), (2048, 9, 1), (700, 90, 6), (200, 40, 16)])
def test_noalloc_planes(n, A, S):
    """The allocation-free Radon on a plan without earlier choices: sizes that its limit admits
    by the one-ray form's workspace."""
    import torch
    from pyraft_amd.device import Plan, current_stream_handle
    from pyraft_amd.raftypes import libraft
    print("radon_noalloc", n, A, S, flush=True)
    p = Plan(n, n, A)
    x = torch.rand(S, n, n, device="cuda")
    out = torch.empty(S, A, n, device="cuda")
    rc = libraft.raft_ss_radon_noalloc(p.handle, ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(out.data_ptr()), 1, 0,
                                       A, S, current_stream_handle(x.device))
    assert rc == 0, libraft.raft_ss_last_error()
    ref = p.radon(x, angle_major=True)
    assert _rel(out.cpu().numpy(), ref.cpu().numpy().astype(np.float64)) <= 1e-6


@pytest.mark.parametrize("sc,S", [((0.0, 1.0, PI, -1.0), 6), ((0.0, 1.0, 2.0, -1.0), 6),
                                  ((0.0, 1.03, PI, -0.97), 8)])
def test_radon_large_values(sc, S):
    """Ray sums near the end of FP32's range stay finite: a block of 1e36 (the sums below 1e38) in
    every kind of planes, launches that take them undivided."""
    import torch
    from pyraft_amd.device import Plan
    n, R, A = 512, 512, 720
    x = np.zeros((n, n), np.float32)
    x[200:280, 220:340] = 1e36
    ref = O.radon(x.astype(np.float64), R, A, **_geo(sc))
    assert 1e35 < np.abs(ref).max() < 1e38
    got = Plan(n, R, A, sino_corners=sc).radon(torch.from_numpy(x).cuda().expand(S, n, n).contiguous()).cpu().numpy()
    assert np.isfinite(got).all()
    for i in (0, 1, S - 1):
        assert _rel(got[i], ref) <= REL


@pytest.mark.parametrize("n,A,sc,S", [(512, 720, (0.0, 1.0, PI, -1.0), 1), (512, 720, (0.0, 1.0, PI, -1.0), 5),
                                      (363, 400, (0.0, 1.0, 2.0, -1.0), 2), (256, 1500, (0.0, 1.0, 2.0, -1.0), 1),
                                      (393, 500, (0.0, 1.0, PI, -1.0), 1)])
def test_transpose_border_pixels(n, A, sc, S):
    """Every pixel, also of the first and last rows and columns: at these sides the float below
    top - eps, where a border candidate's position decides without its range, rounds down, and
    some candidates lie on it.  FP32 weights are within 2e-5 of the exact ones; a sample left
    out is 1e-3 of a pixel's sum and more."""
    import torch
    from pyraft_amd.device import Plan
    y = (1.0 + np.random.default_rng(n).random((n, A))).astype(np.float32)
    ref = O.radon_transpose(y.astype(np.float64), n, **_geo(sc))
    got = Plan(n, n, A, sino_corners=sc).radon_transpose(torch.from_numpy(y).cuda().expand(S, n, A).contiguous())
    for v in got.cpu().numpy():
        assert np.abs(v - ref).max() <= 2e-5 * np.sqrt(np.mean(ref * ref))


CHOICES = r"""
import sys
sys.path.insert(0, %r)
import torch
from pyraft_amd.device import Plan
for n, A in ((256, 180), (700, 300)):
    Plan(n, n, A).radon(torch.rand((n, n), device="cuda"))
torch.cuda.synchronize()
"""


def test_small_radon_keeps_its_candidates(tmp_path):
    """Launches of less than 2^24 updates, where the planes never pay, choose (and time) among the
    one-ray forms alone; larger ones add the planes to all of those."""
    import json
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    path = tmp_path / "tune.json"
    out = subprocess.run([sys.executable, "-c", CHOICES % root], env=dict(os.environ, PYRAFT_AMD_TUNE_CACHE=str(path)),
                         capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    entries = json.loads(path.read_text())["entries"]
    small = {k.split("|")[-3]: v for k, v in entries.items() if "|256|256|180|" in k}
    large = {k.split("|")[-3]: v for k, v in entries.items() if "|700|700|300|" in k}
    assert set(small) == {"radon"} and "planes" in large
    assert sum(t > 0 for t in small["radon"]["times_us"]) == 5  # both shapes in 32-row slabs and whole, 64 rows
    assert large["planes"]["times_us"][1] > 0 and large["planes"]["times_us"][0] > 0


# one angle on either side of the line between undivided and divided launches: few angles at any
# size, more where the tiles fill the chip; two planes and four
@pytest.mark.parametrize("n,A,sc,groups", [
    (40, 23, (0.0, 1.0, PI, -1.0), False), (40, 24, (0.0, 1.0, PI, -1.0), True),
    (512, 56, (0.0, 1.0, PI, -1.0), False), (512, 57, (0.0, 1.0, PI, -1.0), True),
    (789, 40, (0.0, 1.0, 2.0, -1.0), False), (789, 102, (0.0, 1.0, PI, -1.0), False),
    (789, 103, (0.0, 1.0, PI, -1.0), True), (1448, 24, (0.0, 1.0, PI, -1.0), False),
    (135, 118, (0.0, 1.0, PI, -1.0), True), (135, 121, (0.0, 1.0, PI, -1.0), True),
    (256, 155, (0.0, 1.0, PI, -1.0), True), (256, 158, (0.0, 1.0, PI, -1.0), True),
    (500, 56, (0.0, 1.03, PI, -0.97), False)])
def test_backprojection_few_angles(n, A, sc, groups):
    import torch
    from pyraft_amd.device import Plan
    s = np.random.default_rng(n + A).random((3, n, A)).astype(np.float32)
    p = Plan(n, n, A, sino_corners=sc)
    assert (p.info()["bp_groups"] > 1) == groups
    got = p.backprojection(torch.from_numpy(s).cuda()).cpu().numpy()
    one = p.backprojection(torch.from_numpy(s[0]).cuda()).cpu().numpy()
    ref = O.backprojection(s[0].astype(np.float64), n, **_geo(sc))
    assert _rel(one, ref) <= REL and _rel(got[0], ref) <= REL
    assert _rel(got[2], O.backprojection(s[2].astype(np.float64), n, **_geo(sc))) <= REL


# subsets of at least 128 angles on few tiles: 16 waves a block, of 8, 9 and 65 angles each
@pytest.mark.parametrize("n,R,A,sc,S", [(40, 41, 128, (0.0, 1.0, PI, -1.0), 1), (65, 64, 280, (0.0, 0.9, 2.0, -0.84), 2),
                                        (33, 31, 1030, (0.0, 1.0, PI, -0.94), 1)])
def test_osem_weights_many_angles(n, R, A, sc, S):
    test_osem_weights(n, R, A, sc, S)


def test_line_radon_many_slices():
    """Straight angles' blocks of 65535 slices on a wide detector: with them the planes' launch
    would have more threads than a grid dimension holds, so the one-ray form runs."""
    import torch
    from pyraft_amd.device import DdaPlan
    S, R = 65535, 4096
    print("line radon, %d slices, %d rays" % (S, R), flush=True)
    p = DdaPlan(2, R, 4)
    x = torch.rand((S, 2, 2), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    got = p.radon(x)
    for i in (0, S // 2, S - 1):
        own = p.radon(x[i:i + 1])[0]
        assert float(own.abs().max()) > 0.1
        assert float((got[i] - own).abs().max()) <= 1e-5 * float(own.abs().max()), i


def test_transpose_many_slices():
    """More slices than one launch's grid dimension holds blocks for."""
    import torch
    from pyraft_amd.device import Plan
    S = 14000002
    print("transpose, %d slices" % S, flush=True)
    y = torch.rand((S, 2, 1), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    p = Plan(2, 2, 1)
    got = p.radon_transpose(y)
    for i in (0, S // 2, S - 1):
        own = p.radon_transpose(y[i:i + 1])[0]
        assert float(own.abs().max()) > 0.0
        assert float((got[i] - own).abs().max()) <= 1e-5 * float(own.abs().max()), i


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("sc,S", [((0.0, 1.0, PI, -1.0), 6), ((0.0, 1.0, 2.0, -1.0), 6), ((0.0, 1.03, PI, -0.97), 8),
                                  ((0.0, 1.0, PI, -1.0), 12)])
def test_slices_stay_apart(sc, S, bad):
    """A slice of NaN or Inf next to others that share its trajectories, windows and pixels: the
    others' bits don't change, forwards and backwards, and its own values are not finite."""
    import torch
    from pyraft_amd.device import DdaPlan, Plan
    n, R, A = 512, 512, 720
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.rand((S, n, n), device="cuda", generator=gen)
    y = torch.rand((S, R, A), device="cuda", generator=gen)
    ops = []
    for p in (Plan(n, R, A, sino_corners=sc), DdaPlan(n, R, A, sino_corners=sc)):
        ops += [(p.radon, x), (p.radon_transpose, y), (p.backprojection, y)]
    for k, (op, v) in enumerate(ops):
        print("slices apart", sc, S, bad, k, flush=True)
        clean = op(v)
        w = v.clone()
        w[1] = bad
        got = op(w)
        keep = [i for i in range(S) if i != 1]
        assert torch.equal(got[keep], clean[keep]), k
        assert not torch.isfinite(got[1][n // 2, n // 2])
