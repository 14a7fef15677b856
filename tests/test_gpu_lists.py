"""Tile and region lists built from the boxes, at the edges of that build: words of 64 Gaussians, the
limit of the direct walk (4,096 Gaussians; beyond, row lists of 1,024-Gaussian segments), regions with
more than the 2,048 rows laid out in LDS at a time, Gaussians ordered in space (every hit of a region in
a few words) and grids whose tiles or regions are cut off.  The T->G CSR equals the stable sort of the
G->T pairs bit for bit; the region lists and the row table show in the feature gradients (float32 sums
with the 2^-17 split: 1e-4, as the parity tests)."""
import numpy as np
import pytest
import torch

from oracle import g2v_oracle as O
from tests import workloads as W

pytestmark = pytest.mark.gpu

#        n, voxels, variances, ordered in x
CASES = {
    "one": (1, (9, 7, 5), (0.2, 1.0), False),
    "n63": (63, (17, 9, 3), (0.2, 1.0), False),
    "n65": (65, (8, 8, 16), (0.2, 1.0), False),
    "n513_tall": (513, (12, 20, 37), (0.1, 0.6), False),
    "direct_limit": (4096, (33, 30, 7), (0.05, 0.2), True),
    "row_lists": (4097, (33, 30, 7), (0.05, 0.2), False),
    "row_lists_ordered": (5000, (40, 21, 18), (0.05, 0.2), True),
    "many_rows": (5000, (10, 11, 6), (0.3, 1.0), False),
}


@pytest.mark.parametrize("name", list(CASES))
def test_lists(name):
    from CudaGaussianVoxelizer import _C
    n, dims, var, ordered = CASES[name]
    dev = torch.device("cuda")
    vr = (0.0, 0.0, 0.0) + tuple(0.4 * d + 0.1 for d in dims)
    w = W.Workload(name, n, 4, voxel_range=vr, var_range=var, mean_pad=0.5)
    m, o, c, f = W.generate(w, seed=n)
    if ordered:
        k = torch.argsort(m[:, 0])
        m, o, c, f = (t[k].contiguous() for t in (m, o, c, f))
    vs, vrn = np.array(w.voxel_size, np.float32), np.array(vr, np.float32)
    b = O.gaussian_boxes(m.numpy(), c.numpy(), vs, vrn)
    assert b["dims"] == dims
    off, tid, gid = O.g2t_csr(b["tile_lo"], b["tile_hi"], b["tiles"])
    t = O.t2g_csr(tid, gid, int(np.prod(b["tiles"])))
    print(f"[lists] {name} n={n} {dims} pairs={len(tid)}", flush=True)
    out = _C.gaussian_voxelizer_forward(m.to(dev), o.to(dev), c.to(dev), w.voxel_size, vr, f.to(dev))
    assert np.array_equal(out[6].cpu().numpy(), off) and np.array_equal(out[7].cpu().numpy(), tid)
    d = _C.build_t2g(list(w.voxel_size), list(vr), out[2], out[3], out[6], out[7])
    csr = _C._forward(m.to(dev), o.to(dev), c.to(dev), w.voxel_size, vr, f.to(dev), keep_t2g=True)[1]["csr"]
    for k, key in enumerate(("sorted_tiles", "sorted_gauss", "tile_offsets")):
        assert np.array_equal(d[key].cpu().numpy(), t[key]), key
        assert np.array_equal(csr[k].cpu().numpy(), t[key]), key   # the forward's own lists
    g = torch.Generator().manual_seed(1)
    gD, gF = torch.randn(*dims, generator=g), torch.randn(*dims, 4, generator=g)
    res = _C.gaussian_voxelizer_backward(gD.to(dev), gF.to(dev), m.to(dev), o.to(dev), out[1], w.voxel_size, vr, out[2],
                                         out[3], out[4], out[6], out[7], out[0], out[5], f.to(dev))
    ref = O.backward_f64(gD.numpy(), gF.numpy(), m.numpy(), o.numpy(), c.numpy(), f.numpy(), b["lb"], b["ub"], vs, vrn,
                         density=out[0].cpu().numpy(), grid_feats=out[5].cpu().numpy())
    assert O.rel_err(res[3].cpu().numpy(), ref[3]) < 1e-4


# Few regions and many Gaussians: a region's rows are one workgroup's chain, so beyond a number of rows the pairs are
# sorted, the tiles' (T->G) and the regions' (feature backward) each by its own count.  On either side of both switches:
#        n, voxels, variances, tiles sorted, regions sorted
ROUTES = {
    "four_regions_2000": (2000, (16, 16, 8), (0.1, 0.6), False, False),
    "four_regions_8000": (8000, (16, 16, 8), (0.1, 0.6), True, True),
    "direct_4096_wide": (4096, (16, 16, 8), (0.5, 2.5), True, True),
    "regions_only_7500": (7500, (40, 40, 16), (0.5, 2.5), False, True),
    "row_lists_5000": (5000, (40, 40, 16), (0.1, 0.6), False, False),
}


@pytest.mark.parametrize("name", list(ROUTES))
def test_list_routes(name):
    from CudaGaussianVoxelizer import _C, _lib
    from oracle import g2v_oracle_c as OC
    n, dims, var, tiles_sorted, regions_sorted = ROUTES[name]
    dev = torch.device("cuda")
    vr = (0.0, 0.0, 0.0) + tuple(0.4 * d + 0.1 for d in dims)
    w = W.Workload(name, n, 4, voxel_range=vr, var_range=var)
    m, o, c, f = W.generate(w, seed=n)
    vs, vrn = np.array(w.voxel_size, np.float32), np.array(vr, np.float32)
    b = O.gaussian_boxes(m.numpy(), c.numpy(), vs, vrn)
    off, tid, gid, toff, sg = OC.csr(b["tile_lo"], b["tile_hi"], b["tiles"])
    print(f"[routes] {name} n={n} {dims} pairs={len(tid)}", flush=True)

    def kernels(call):
        _lib.profile_reset()
        _lib.profile_enable(True)
        try:
            out = call()
            torch.cuda.synchronize()
            return out, " ".join(_lib.profile_report())
        finally:
            _lib.profile_enable(False)
            _lib.profile_reset()

    out, ran = kernels(lambda: _C.gaussian_voxelizer_forward(m.to(dev), o.to(dev), c.to(dev), w.voxel_size, vr, f.to(dev)))
    assert ("k_fill_g2t" in ran) == ("k_radix_scatter" in ran) == tiles_sorted, ran
    g = torch.Generator().manual_seed(1)
    gD, gF = torch.randn(*dims, generator=g), torch.randn(*dims, 4, generator=g)
    res, ran = kernels(lambda: _C.gaussian_voxelizer_backward(
        gD.to(dev), gF.to(dev), m.to(dev), o.to(dev), out[1], w.voxel_size, vr, out[2], out[3], out[4], out[6], out[7],
        out[0], out[5], f.to(dev)))
    assert ("k_fill_cells" in ran) == regions_sorted, ran
    Ainv = np.linalg.inv(c.numpy().reshape(-1, 3, 3).astype(np.float64)).reshape(-1, 9)
    D, F = OC.forward(m.numpy(), o.numpy(), Ainv, b["lb"], b["ub"], vs, vrn, toff, sg, f.numpy(), b["dims"])
    assert O.rel_err(out[0].cpu().numpy(), D) < 1e-4 and O.rel_err(out[5].cpu().numpy(), F) < 1e-4
    ref = OC.backward(m.numpy(), o.numpy(), Ainv, b["lb"], b["ub"], vs, vrn, off, tid, f.numpy(), out[0].cpu().numpy(),
                      out[5].cpu().numpy(), gD.numpy(), gF.numpy())
    assert O.rel_err(res[3].cpu().numpy(), ref[3]) < 1e-4


@pytest.mark.parametrize("n,dims", [(600, (17, 9, 7)), (5000, (40, 40, 16)), (9000, (16, 16, 8))])
def test_build_t2g_sorts_the_given_ids(n, dims):
    """build_t2g is the stable sort of the ids it is given, also where they are not those of the boxes."""
    from CudaGaussianVoxelizer import _C
    dev = torch.device("cuda")
    vr = (0.0, 0.0, 0.0) + tuple(0.4 * d + 0.1 for d in dims)
    w = W.Workload("ids", n, None, voxel_range=vr, var_range=(0.1, 0.6))
    m, o, c, _ = W.generate(w, seed=n)
    out = _C.gaussian_voxelizer_forward(m.to(dev), o.to(dev), c.to(dev), w.voxel_size, vr)
    T = int(np.prod([-(-d // 4) for d in dims]))
    off, tid = out[6].cpu().numpy(), T - 1 - out[7].cpu().numpy()
    d = _C.build_t2g(list(w.voxel_size), list(vr), out[2], out[3], out[6], torch.from_numpy(tid).to(dev))
    t = O.t2g_csr(tid, np.repeat(np.arange(n, dtype=np.int32), np.diff(off)), T)
    for key in ("sorted_tiles", "sorted_gauss", "tile_offsets", "unique_tiles", "counts"):
        assert np.array_equal(d[key].cpu().numpy(), t[key]), key
