"""GPU parity of the 3D projector (slice and general modes) against the
oracle, through the C ABI.

Bar: ul indices and the four weights bit-exact; projections and back
projections within rel-L2 1e-5 of the float32 oracle; dot test <= 1e-5;
the reference's known-answer arrays (test_xray_3d.py:29-69).  The full
256^3 / 360-view case is checked slice by slice against the oracle on thin
volumes (slices are independent for a single rotation axis) plus the dot
test and per-view mass.
"""

import json
import os

import numpy as np
import pytest
import torch

from oracle import xray as X
from scico_amd import phantom
from scico_amd.linop import valid_adjoint
from scico_amd.linop.xray import XRayTransform3D
from tests.conftest import rel_l2

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden")


def _mats(shape, det, seq, ang, **kw):
    return XRayTransform3D.matrices_from_euler_angles(shape, det, seq, ang, **kw)


# (shape, det, seq, angles, kwargs, expected mode)
GEOMS = [
    ((16, 16, 16), (24, 16), "Y", np.linspace(0, np.pi, 12, endpoint=False), {}, "slice"),
    ((9, 7, 5), (14, 7), "Y", np.linspace(0, np.pi, 7, endpoint=False), {}, "slice"),
    ((8, 6, 10), (14, 10), "Y", np.linspace(0, np.pi, 5, endpoint=False), {}, "slice"),  # det != S
    ((6, 11, 13), (12, 18), "X", np.linspace(0, np.pi, 6, endpoint=False)[:, None], {}, "slice"),
    ((6, 11, 13), (11, 18), "X", np.linspace(0, np.pi, 6, endpoint=False)[:, None], {}, "general"),
    ((12, 10, 8), (16, 14), "Z", np.linspace(0, np.pi, 6, endpoint=False), {}, "general"),
    ((8, 6, 9), (13, 9), "Y", np.linspace(0, np.pi, 4, endpoint=False), {}, "general"),  # t_d = 1/4
    ((10, 9, 8), (16, 16), "XYZ",
     np.random.default_rng(0).uniform(0, np.pi, (5, 3)), {}, "general"),
    ((8, 8, 8), (12, 12), "Y", np.linspace(0, np.pi, 5, endpoint=False),
     {"voxel_spacing": [1.0, 1.0, 1.5]}, "slice"),
]


def _op(shape, det, seq, ang, kw, allow_slice=True):
    M = _mats(shape, det, seq, ang, **kw)
    H = XRayTransform3D(shape, M, det)
    H._allow_slice = allow_slice
    return H, H.matrices


@pytest.mark.parametrize("g", range(len(GEOMS)))
def test_mode_selection(gpu, g):
    shape, det, seq, ang, kw, mode = GEOMS[g]
    H, _ = _op(shape, det, seq, ang, kw)
    assert H.info()["mode"] == mode


@pytest.mark.parametrize("allow_slice", [True, False])
@pytest.mark.parametrize("g", range(len(GEOMS)))
def test_weights_bit_exact(gpu, g, allow_slice):
    shape, det, seq, ang, kw, _ = GEOMS[g]
    H, M = _op(shape, det, seq, ang, kw, allow_slice)
    for v in range(len(M)):
        ul, w = H.weights(v)
        rul, *rw = X.calc_weights_3d(shape, M[v], det)
        np.testing.assert_array_equal(ul.cpu().numpy(), rul)
        np.testing.assert_array_equal(w.cpu().numpy(), np.stack(rw))


@pytest.mark.parametrize("allow_slice", [True, False])
@pytest.mark.parametrize("g", range(len(GEOMS)))
def test_forward_adjoint_parity(gpu, g, allow_slice):
    shape, det, seq, ang, kw, _ = GEOMS[g]
    H, M = _op(shape, det, seq, ang, kw, allow_slice)
    print(f"xr3d {shape} {det} {seq} mode={H.info()['mode']}", flush=True)
    rng = np.random.default_rng(g)
    x = rng.random(shape).astype(np.float32)
    y = rng.standard_normal(H.output_shape).astype(np.float32)
    e_f = rel_l2(H(x).cpu().numpy(), X.project_3d(x, M, det))
    e_a = rel_l2(H.T(y).cpu().numpy(), X.back_project_3d(y, M, shape))
    print(f"  rel-L2 fwd {e_f:.2e} adj {e_a:.2e}", flush=True)
    assert e_f <= 1e-5 and e_a <= 1e-5
    assert valid_adjoint(H, H.T, eps=1e-5)


def test_reference_kat(gpu):
    """test_xray_3d.py:29-69 known-answer arrays, both modes."""
    kat = json.load(open(os.path.join(GOLD, "reference_kat.json")))["xray3d_scaling"]
    x = np.zeros(kat["input_shape"], np.float32)
    s = kat["ones_slice"]
    x[s[0][0] : s[0][1], s[1][0] : s[1][1], s[2][0] : s[2][1]] = 1
    for case in kat["cases"]:
        M = XRayTransform3D.matrices_from_euler_angles(
            x.shape, x.shape[:2], kat["seq"], kat["angles"], voxel_spacing=case["voxel_spacing"])
        for allow in (True, False):
            H = XRayTransform3D(x.shape, matrices=M, det_shape=x.shape[:2])
            H._allow_slice = allow
            np.testing.assert_allclose(H(x).cpu().numpy(), np.array(case["truth"]), atol=1e-6)


def test_matched_adjoint(gpu):
    """test_xray_3d.py:9-26."""
    N = 16
    dc = int(N * 1.05 / np.sqrt(2.0))
    M = XRayTransform3D.matrices_from_euler_angles(
        (N, N, N), (dc, dc), "X", np.linspace(0, np.pi, 3, endpoint=False)[:, None])
    H = XRayTransform3D((N, N, N), matrices=M, det_shape=(dc, dc))
    assert valid_adjoint(H, H.T, eps=1e-5)


def test_determinism_slice_mode(gpu):
    shape, det = (32, 24, 40), (48, 24)
    H, _ = _op(shape, det, "Y", np.linspace(0, np.pi, 30, endpoint=False), {})
    x = torch.rand(shape, device="cuda")
    y1, y2 = H(x), H(x)
    b1, b2 = H.T(y1), H.T(y1)
    assert torch.equal(y1, y2) and torch.equal(b1, b2)


def test_full_size_256_360(gpu):
    """256^3 volume, 360 views about axis 1, detector 368 x 256: slices
    {0, 77, 255} against the oracle on thin volumes, per-view mass, dot
    test."""
    N, V, det = 256, 360, (368, 256)
    ang = phantom.angles(V)
    M = XRayTransform3D.matrices_from_euler_angles((N, N, N), det, "Y", ang)
    H = XRayTransform3D((N, N, N), M, det)
    assert H.info()["mode"] == "slice" and H.info()["projection_in_place"]
    vol = phantom.ellipsoid_phantom((N, N, N), 30, seed=0)
    y = H(vol)
    yn = y.cpu().numpy()
    sub = np.arange(0, V, 18)
    Mt = X.matrices_from_euler_angles((N, 1, N), (det[0], 1), "Y", ang)
    rng = np.random.default_rng(3)
    yr = rng.standard_normal((V, *det)).astype(np.float32)
    bp = H.T(yr).cpu().numpy()
    for j in (0, 77, 255):
        thin = np.ascontiguousarray(vol[:, j : j + 1, :])
        ref = X.project_3d(thin, Mt[sub].astype(np.float32), (det[0], 1))[..., 0]
        e = rel_l2(yn[sub, :, j], ref)
        ref_bp = X.back_project_3d(np.ascontiguousarray(yr[:, :, j : j + 1]),
                                   Mt.astype(np.float32), (N, 1, N))[:, 0, :]
        eb = rel_l2(bp[:, j, :], ref_bp)
        print(f"  256^3/360 slice {j}: fwd rel-L2 {e:.2e}, adj rel-L2 {eb:.2e}", flush=True)
        assert e <= 1e-5 and eb <= 1e-5
    # every footprint is on the detector: each view carries the volume's mass
    sums = y.double().sum(dim=(1, 2)).cpu().numpy()
    np.testing.assert_allclose(sums, np.full(V, vol.astype(np.float64).sum()), rtol=1e-5)
    assert valid_adjoint(H, H.T, eps=1e-5)


STAGED_CASES = [g for g in range(len(GEOMS)) if GEOMS[g][5] == "slice"] + ["full", "slab"]


@pytest.mark.parametrize("case", STAGED_CASES)
def test_staged_adjoint_bitwise(gpu, case):
    """The slice adjoint that copies each view's detector rows for a 4 x 8
    pixel tile into LDS equals the one that reads them from global memory,
    bit for bit (same rows, same accumulation order); plans whose tile
    range can exceed the staging buffer keep the global-memory kernel."""
    if case == "full":
        shape, det, seq, ang, kw = (256, 256, 256), (368, 256), "Y", phantom.angles(360), {}
    elif case == "slab":
        shape, det, seq, ang, kw = (256, 16, 256), (368, 16), "Y", phantom.angles(360), {}
    else:
        shape, det, seq, ang, kw, _ = GEOMS[case]
    H, _ = _op(shape, det, seq, ang, kw)
    Hg, _ = _op(shape, det, seq, ang, kw)
    Hg._stage_adjoint = False
    assert H.info()["mode"] == "slice" and not Hg.info()["adjoint_staged"]
    y = torch.randn(H.output_shape, device="cuda",
                    generator=torch.Generator("cuda").manual_seed(11))
    staged = H.info()["adjoint_staged"]
    print(f"  staged adjoint {shape} {det} views {len(ang)}: staged={staged}", flush=True)
    if case in ("full", "slab"):
        assert staged
    assert torch.equal(H.T(y), Hg.T(y))


def _tilted(shape, det, seq, n, **kw):
    ang = np.stack(np.broadcast_arrays(74.0, np.linspace(0, 180, n, endpoint=False)), axis=-1)
    return _mats(shape, det, seq, ang, degrees=True, **kw)


# (shape, det, matrices): blocks of the splat are 24 voxels, of the adjoint 8;
# march axes x, y and z; detectors smaller and larger than the object; few
# and many views; other voxel spacings (other lane strides); spacings whose
# windows do not fit (the gathers)
WINDOW_CASES = {
    "tilt": ((33, 30, 31), (40, 42), lambda s, d: _tilted(s, d, "XY", 5)),
    "one_voxel": ((1, 1, 1), (3, 3), lambda s, d: _tilted(s, d, "XY", 3)),
    "edges": ((24, 8, 25), (16, 17), lambda s, d: _tilted(s, d, "XY", 4)),
    "march_z": ((17, 49, 40), (60, 31), lambda s, d: _mats(
        s, d, "XY", np.random.default_rng(1).uniform(-0.3, 0.3, (4, 2)))),
    "march_x": ((47, 26, 23), (33, 50), lambda s, d: _mats(
        s, d, "YX", np.pi / 2 + np.random.default_rng(2).uniform(-0.3, 0.3, (4, 2)))),
    "any": ((40, 28, 36), (48, 48), lambda s, d: _mats(
        s, d, "XYZ", np.random.default_rng(3).uniform(0, np.pi, (70, 3)))),
    "fine": ((40, 40, 40), (24, 24), lambda s, d: _tilted(s, d, "XY", 4,
                                                          voxel_spacing=[0.6, 0.6, 0.6])),
    "stretched": ((20, 24, 18), (40, 40), lambda s, d: _tilted(s, d, "XY", 4,
                                                               voxel_spacing=[1.0, 1.3, 0.8])),
    "too_wide": ((12, 12, 12), (64, 64), lambda s, d: _tilted(s, d, "XY", 3,
                                                              voxel_spacing=[4.0, 4.0, 4.0])),
}


@pytest.mark.parametrize("case", list(WINDOW_CASES))
def test_general_windows(gpu, case):
    """General-mode projections through detector windows in LDS against the
    oracle and the gathers from global memory (sums of the same terms in
    another order: a few float32 roundings of relative size 6e-8 each, as
    the bars of the other parity tests); twice the same bits; into an output
    that is not 16-byte aligned; and on a side stream while the default
    stream projects another volume with the same operator."""
    shape, det, mk = WINDOW_CASES[case]
    M = mk(shape, det)
    H = XRayTransform3D(shape, M, det)
    G = XRayTransform3D(shape, M, det)
    G._windows = False
    assert H.info()["mode"] == "general"
    rng = np.random.default_rng(11)
    x = torch.as_tensor(rng.random(shape).astype(np.float32), device="cuda")
    y = torch.as_tensor(rng.standard_normal(H.output_shape).astype(np.float32), device="cuda")
    p, b = H(x), H.adj(y)
    e = (rel_l2(p.cpu(), X.project_3d(x.cpu().numpy(), H.matrices, det)),
         rel_l2(b.cpu(), X.back_project_3d(y.cpu().numpy(), H.matrices, shape)),
         rel_l2(p.cpu(), G(x).cpu()), rel_l2(b.cpu(), G.adj(y).cpu()))
    print(f"  {case}: oracle fwd {e[0]:.2e} adj {e[1]:.2e}, gathers fwd {e[2]:.2e} adj {e[3]:.2e}",
          flush=True)
    assert max(e) <= 1e-5
    assert torch.equal(p, H(x)) and torch.equal(b, H.adj(y))
    off = torch.empty(b.numel() + 1, device="cuda")[1:]
    assert torch.equal(H.back_project(y, out=off).reshape(shape), b)
    off = torch.empty(p.numel() + 1, device="cuda")[1:]
    assert torch.equal(H.project(x, out=off).reshape(p.shape), p)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        ps = [H(x) for _ in range(4)]
    pd = [H(2.0 * x) for _ in range(4)]
    torch.cuda.synchronize()
    assert all(torch.equal(q, p) for q in ps) and all(torch.equal(q, 2.0 * p) for q in pd)


@pytest.mark.parametrize("shape,views,scale,shift", [
    ((1, 4, 1), 2, 1.0, 0.0),  # one pixel
    ((5, 4, 9), 3, 1.0, 0.0),  # rows no multiple of 4, bins no multiple of 7
    ((33, 12, 20), 6, 1.0, -7.3),  # strip partly off the detector
    ((16, 260, 16), 5, 1.0, 0.0),  # more than 64 slice quads
    ((21, 8, 30), 9, 0.945, 2.5),  # spacing just above and just below the limit of
    ((21, 8, 30), 9, 0.942, 2.5),  # 16 candidates in a row
    ((24, 8, 24), 8, 1.3, 0.0),  # wide spacing: empty bin groups
    ((24, 8, 24), 8, 0.72, 0.0),  # three pixels in a bin group
])
def test_slice_strips(gpu, shape, views, scale, shift):
    """Slice-mode forward and adjoint against float64 sums of the operator's
    own weights, over the forms of the forward's strips; n products added in
    float32 are off by at most n eps times the absolute sum."""
    th = np.linspace(0, np.pi, views, endpoint=False)
    rows = np.zeros((views, 2, 3))
    rows[:, 0, 0], rows[:, 0, 2] = scale * np.cos(th), scale * np.sin(th)
    rows[:, 1, 1] = 1.0
    det = (int(np.ceil(scale * np.hypot(shape[0], shape[2]))) + 1, shape[1])
    t = np.asarray(det) / 2 - rows @ (np.asarray(shape) / 2)
    t[:, 0] += shift
    H = XRayTransform3D(shape, np.concatenate((rows, t[..., None]), axis=2), det)
    assert H.info()["mode"] == "slice"
    rng = np.random.default_rng(3)
    x = rng.standard_normal(shape).astype(np.float32)
    y = rng.standard_normal(H.output_shape).astype(np.float32)
    fwd = H.project(torch.as_tensor(x, device="cuda")).cpu().numpy()
    adj = H.back_project(torch.as_tensor(y, device="cuda")).cpu().numpy()
    ref = np.zeros((3, views, det[0] + 2, det[1]))  # sum, absolute sum, products
    back = np.zeros((2, *shape))
    for v in range(views):
        ul, w = (a.cpu().numpy() for a in H.weights(v))
        at1 = np.clip(ul[1], 0, det[1] - 1)
        for k in (0, 1):  # detector rows ul and ul + 1 (the slice axis has one tap)
            at0 = np.clip(ul[0] + k, -1, det[0]) + 1
            prod = x.astype(np.float64) * w[k]
            np.add.at(ref[0, v], (at0, at1), prod)
            np.add.at(ref[1, v], (at0, at1), np.abs(prod))
            np.add.at(ref[2, v], (at0, at1), 1)
            yv = np.pad(y[v].astype(np.float64), ((1, 1), (0, 0)))[at0, at1]
            back[0] += yv * w[k]
            back[1] += np.abs(yv * w[k])
    eps = 2.0**-24
    assert np.all(np.abs(fwd - ref[0, :, 1:-1]) <= eps * (ref[2] * ref[1])[:, 1:-1] + 1e-30)
    assert np.all(np.abs(adj - back[0]) <= eps * 2 * views * back[1] + 1e-30)


@pytest.mark.parametrize("case", list(WINDOW_CASES))
def test_general_windows_small(gpu, case):
    """The kernels with windows in LDS on volumes so small that the gathers
    are the default: against the gathers (bar as in test_general_windows)."""
    shape, det, mk = WINDOW_CASES[case]
    M = mk(shape, det)
    H, G = XRayTransform3D(shape, M, det), XRayTransform3D(shape, M, det)
    H._windows, G._windows = "always", False
    rng = np.random.default_rng(12)
    x = torch.as_tensor(rng.random(shape).astype(np.float32), device="cuda")
    y = torch.as_tensor(rng.standard_normal(H.output_shape).astype(np.float32), device="cuda")
    e = rel_l2(H(x).cpu(), G(x).cpu()), rel_l2(H.adj(y).cpu(), G.adj(y).cpu())
    assert max(e) <= 1e-5 and H._ws_floats > 0 and G._ws_floats == 0


@pytest.mark.parametrize("shape,det,views,splat", [
    ((16, 16, 16), (24, 16), 1, False), ((23, 24, 25), (40, 42), 4, False),
    ((66, 66, 66), (74, 66), 40, True), ((96, 96, 96), (120, 120), 3, True),
    ((32, 32, 32), (500, 500), 3, True), ((256, 256, 1), (300, 300), 4, True)])
def test_general_windows_rule(gpu, shape, det, views, splat):
    """The default takes the forward's windows where the gather has more to
    do, and is the path that it takes, bit for bit."""
    M = _tilted(shape, det, "XY", views)
    H = XRayTransform3D(shape, M, det)
    W = XRayTransform3D(shape, M, det)
    H._allow_slice = W._allow_slice = False
    W._windows = "always" if splat else False
    x = torch.as_tensor(np.random.default_rng(5).random(shape).astype(np.float32), device="cuda")
    assert torch.equal(H(x), W(x)) and (H._ws_floats > 0) == splat


def test_general_forward_without_memory(gpu, monkeypatch):
    """No memory for the windows: the forward is the gather's, bit for bit."""
    from scico_amd.linop.xray import _xray3d

    shape, det, mk = WINDOW_CASES["any"]
    H, G = (XRayTransform3D(shape, mk(shape, det), det) for _ in range(2))
    G._windows = False
    x = torch.as_tensor(np.random.default_rng(6).random(shape).astype(np.float32), device="cuda")
    ref, out = G(x), torch.empty(H.output_shape, device="cuda")
    assert H.plan and H._ws_floats > 0

    def empty(shape, dtype=np.float32):
        raise torch.OutOfMemoryError("no memory")

    monkeypatch.setattr(_xray3d.dev, "empty", empty)
    assert torch.equal(H.project(x, out=out), ref)
