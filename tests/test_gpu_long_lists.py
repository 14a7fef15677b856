"""Tiles with long lists (phase A's passes of 256 Gaussians on the bfloat16 matrix cores) at the edges of
their blocks: lists around one block of 32 entries, one pass (256) and two, channel counts that give 1 to 7
chunks (the chunk loop takes three at a time) with and without 16-byte rows, and a grid that no tile
divides; and phase B's two shapes (rows of up to 64 channels and wider ones) around their passes of 320 and
384 region rows.

Every Gaussian covers the whole grid, so every tile's list holds all of them.  The split leaves 2^-17 =
7.6e-6 of each product and the float32 sums of at most 520 terms less than 520 * 2^-24 = 3.1e-5 of the sum of the
terms' magnitudes (in the mean over the voxels far less: the roundings are of either sign).  Densities and
features: 3e-5; the feature gradients, sums of either sign over the voxels, 3e-5 of the sums of magnitudes.
The gradients of the geometry are differences (u - t) of such sums, amplified by the cancellation between them:
3e-4.  A bfloat16 output is the float value rounded (2^-9)."""
import numpy as np
import pytest
import torch

from oracle import g2v_oracle as O

pytestmark = pytest.mark.gpu

VS, VR = (0.4, 0.4, 0.4), (0.0, 0.0, 0.0, 2.0, 2.8, 2.4)   # 5 x 7 x 6 voxels (2.4 / 0.4 truncates to 6 or 5)


def _scene(n, C, seed):
    g = torch.Generator().manual_seed(seed)
    m = torch.rand(n, 3, generator=g) * torch.tensor([2.0, 2.8, 2.4])
    q, _ = torch.linalg.qr(torch.randn(n, 3, 3, generator=g))
    var = torch.rand(n, 3, generator=g) * 2.0 + 2.0       # 3 sigma > the grid's diagonal extent per axis
    cov = (q @ torch.diag_embed(var) @ q.mT).reshape(n, 9).contiguous()
    return m, torch.rand(n, generator=g) + 0.1, cov, torch.randn(n, C, generator=g)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,C", [(65, 1), (65, 32), (96, 64), (97, 97), (128, 128), (129, 161), (160, 260), (255, 200),
                                 (256, 224), (257, 96), (300, 33), (520, 36), (321, 64), (320, 63), (385, 66), (33, 384), (225, 448)])
def test_long_lists(n, C, dtype):
    from CudaGaussianVoxelizer import _C
    dev = torch.device("cuda")
    m, o, c, f = _scene(n, C, seed=n + C)
    f = f.to(dtype)
    vs, vr = np.array(VS, np.float32), np.array(VR, np.float32)
    b = O.gaussian_boxes(m.numpy(), c.numpy(), vs, vr)
    assert (b["ntiles"] == np.prod(b["tiles"])).all()
    out = _C.gaussian_voxelizer_forward(m.to(dev), o.to(dev), c.to(dev), VS, VR, f.to(dev))
    X, Y, Z = b["dims"]
    g = torch.Generator().manual_seed(3)
    gD, gF = torch.randn(X, Y, Z, generator=g), torch.randn(X, Y, Z, C, generator=g).to(dtype)
    res = _C.gaussian_voxelizer_backward(gD.to(dev), gF.to(dev), m.to(dev), o.to(dev), out[1], VS, VR, out[2], out[3],
                                         out[4], out[6], out[7], out[0], out[5], f.to(dev))
    f64, gF64 = f.double().numpy(), gF.double().numpy()
    D, F = O.forward_f64(m.numpy(), o.numpy(), c.numpy(), f64, b["lb"], b["ub"], vs, vr)
    ref = O.backward_f64(gD.numpy(), gF64, m.numpy(), o.numpy(), c.numpy(), f64, b["lb"], b["ub"], vs, vr)
    mag = O.backward_f64(gD.numpy(), np.abs(gF64), m.numpy(), o.numpy(), c.numpy(), f64, b["lb"], b["ub"], vs, vr)[3]
    feat, tol = (3e-5, 3e-4) if dtype == torch.float32 else (2.0 ** -9, 2e-3)
    err = {"density": (O.rel_err(out[0].cpu().numpy(), D), 3e-5),
           "grid_feats": (O.rel_err(out[5].float().cpu().numpy(), F), feat),
           "features": (np.linalg.norm(res[3].float().cpu().numpy() - ref[3]) / np.linalg.norm(mag), feat),
           "means": (O.rel_err(res[0].cpu().numpy(), ref[0]), tol), "cov": (O.rel_err(res[1].cpu().numpy(), ref[1]), tol),
           "opacity": (O.rel_err(res[2].cpu().numpy(), ref[2]), tol)}
    print(f"[long] n={n} C={C} {dtype}: " + ", ".join(f"{k} {v:.1e}" for k, (v, _) in err.items()), flush=True)
    for k, (v, t) in err.items():
        assert v < t, (k, v, t)


@pytest.mark.parametrize("C,dtype", [(16, torch.float32), (33, torch.float32), (64, torch.bfloat16)])
def test_many_regions_of_long_rows(C, dtype):
    """Rows of at most 64 channels in more regions than run at once (23 x 23), whose lists are too long for one pass of
    phase B's narrow shape and fit one of the wide shape's: the wide shape.  A feature gradient's float32 sums run over at most 1,024 voxels of a region and 49 regions: 3e-5 of
    the sums of magnitudes, as above."""
    from CudaGaussianVoxelizer import _C
    from oracle import g2v_oracle_c as OC
    from tests import workloads as W
    from tests.test_gpu_lists import kernels
    dev = torch.device("cuda")
    w = W.Workload("long_rows", 5500, C, voxel_range=(0.0, 0.0, 0.0, 73.7, 73.7, 1.7), var_range=(2.0, 12.0))
    m, o, c, f = W.generate(w, seed=C)
    f = f.to(dtype)
    vs, vr = np.array(w.voxel_size, np.float32), np.array(w.voxel_range, np.float32)
    b = O.gaussian_boxes(m.numpy(), c.numpy(), vs, vr)
    assert b["dims"] == (184, 184, 4)
    rows = ((b["ub"][:, :2] // 8 - b["lb"][:, :2] // 8 + 1).prod(1) * (b["nvox"] > 0)).sum()
    assert 320 < rows * 1.15 / 23 ** 2 < 384
    print(f"[rows] C={C} {dtype} {rows} rows", flush=True)
    out = _C.gaussian_voxelizer_forward(m.to(dev), o.to(dev), c.to(dev), w.voxel_size, w.voxel_range, f.to(dev))
    X, Y, Z = b["dims"]
    g = torch.Generator().manual_seed(3)
    gD, gF = torch.zeros(X, Y, Z), torch.randn(X, Y, Z, C, generator=g).to(dtype)
    res, ran = kernels(lambda: _C.gaussian_voxelizer_backward(
        gD.to(dev), gF.to(dev), m.to(dev), o.to(dev), out[1], w.voxel_size, w.voxel_range, out[2], out[3], out[4],
        out[6], out[7], out[0], out[5], f.to(dev)))
    assert "k_bwd_region" in ran and "BrNarrow" not in ran, ran
    off, tid, gid, toff, sg = OC.csr(b["tile_lo"], b["tile_hi"], b["tiles"])
    Ainv = np.linalg.inv(c.numpy().reshape(-1, 3, 3).astype(np.float64)).reshape(-1, 9)

    def grad(up):
        return OC.backward(m.numpy(), o.numpy(), Ainv, b["lb"], b["ub"], vs, vr, off, tid, f.float().numpy(),
                           out[0].cpu().numpy(), out[5].float().cpu().numpy(), gD.numpy(), up)[3]

    gF32 = gF.float().numpy()
    err = np.linalg.norm(res[3].float().cpu().numpy() - grad(gF32)) / np.linalg.norm(grad(np.abs(gF32)))
    assert err < (3e-5 if dtype == torch.float32 else 2.0 ** -9), err


@pytest.mark.parametrize("n,dims,C", [(5000, (16, 16, 4), 4), (5000, (16, 16, 4), 5), (1500, (32, 32, 16), 4)])
def test_few_tiles_of_many_passes(n, dims, C):
    """Up to 256 tiles, the passes of phase A over a tile's list are split over workgroups: 20 passes over 16, and 6
    over 2.  The float32 sums of each pair are the same as in one workgroup; features and geometry as above."""
    from CudaGaussianVoxelizer import _C
    from oracle import g2v_oracle_c as OC
    from tests import workloads as W
    dev = torch.device("cuda")
    w = W.Workload("few", n, C, voxel_range=(0.0, 0.0, 0.0) + tuple(0.4 * d + 0.1 for d in dims), var_range=(8.0, 20.0))
    m, o, c, f = W.generate(w, seed=n + C)
    vs, vr = np.array(w.voxel_size, np.float32), np.array(w.voxel_range, np.float32)
    b = O.gaussian_boxes(m.numpy(), c.numpy(), vs, vr)
    assert b["dims"] == dims
    off, tid, gid, toff, sg = OC.csr(b["tile_lo"], b["tile_hi"], b["tiles"])
    print(f"[few] n={n} {dims} lists {np.diff(toff).min()} to {np.diff(toff).max()}", flush=True)
    out = _C.gaussian_voxelizer_forward(m.to(dev), o.to(dev), c.to(dev), w.voxel_size, w.voxel_range, f.to(dev))
    g = torch.Generator().manual_seed(3)
    gD, gF = torch.randn(*dims, generator=g), torch.randn(*dims, C, generator=g)
    res = _C.gaussian_voxelizer_backward(gD.to(dev), gF.to(dev), m.to(dev), o.to(dev), out[1], w.voxel_size,
                                         w.voxel_range, out[2], out[3], out[4], out[6], out[7], out[0], out[5], f.to(dev))
    Ainv = np.linalg.inv(c.numpy().reshape(-1, 3, 3).astype(np.float64)).reshape(-1, 9)

    def grad(gd, up):
        return OC.backward(m.numpy(), o.numpy(), Ainv, b["lb"], b["ub"], vs, vr, off, tid, f.numpy(),
                           out[0].cpu().numpy(), out[5].cpu().numpy(), gd, up)

    ref, mag = grad(gD.numpy(), gF.numpy()), grad(gD.numpy(), np.abs(gF.numpy()))[3]
    assert np.linalg.norm(res[3].cpu().numpy() - ref[3]) / np.linalg.norm(mag) < 3e-5
    for k, what in ((0, "means"), (1, "cov"), (2, "opacity")):
        assert O.rel_err(res[k].cpu().numpy(), ref[k]) < 3e-4, what
