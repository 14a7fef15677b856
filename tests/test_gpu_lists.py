"""Tile and region lists built from the boxes, at the edges of that build: words of 64 Gaussians, the
limit of the direct walk (4,096 Gaussians; beyond, row lists of 1,024-Gaussian segments), regions with
more than the 2,048 rows laid out in LDS at a time, Gaussians ordered in space (every hit of a region in
a few words) and grids whose tiles or regions are cut off; and the sorted build beyond the rules' limits, alone
and in batches.  The T->G CSR equals the stable sort of the
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
    "many_rows": (5000, (10, 11, 6), (0.3, 1.0), False),   # sorted: 2,842 to 4,999 rows in each of four regions
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


def kernels(call):
    """The call's result and the names of the library's kernels that it launched."""
    from CudaGaussianVoxelizer import _lib
    _lib.profile_reset()
    _lib.profile_enable(True)
    try:
        out = call()
        torch.cuda.synchronize()
        return out, " ".join(_lib.profile_report())
    finally:
        _lib.profile_enable(False)
        _lib.profile_reset()


# Few regions and many Gaussians: a region's rows are one workgroup's chain, so beyond a number of rows the pairs are
# sorted, the tiles' (T->G) and the regions' (feature backward) each by its own count.  On either side of both switches:
#        n, voxels, variances, tiles sorted, regions sorted
ROUTES = {
    "four_regions_2000": (2000, (16, 16, 8), (0.1, 0.6), False, False),
    "four_regions_8000": (8000, (16, 16, 8), (0.1, 0.6), True, True),
    "direct_4096_wide": (4096, (16, 16, 8), (0.5, 2.5), True, True),
    "regions_only_7500": (7500, (40, 40, 16), (0.5, 2.5), False, True),
    "row_lists_5000": (5000, (40, 40, 16), (0.1, 0.6), False, False),
    # 33,125 visits of the direct walk: everything is sorted
    "many_visits_3329": (3329, (200, 200, 16), (0.1, 0.6), True, True),
    # 20,800 tiles: the lists' offsets are scanned, not summed by the workgroups
    "scanned_offsets_1000": (1000, (160, 160, 52), (0.3, 1.5), False, False),
    # regions of more than the 2,048 rows laid out at a time, in the direct walk and (all Gaussians about four
    # regions, which the mean does not show) with row lists
    "row_chunks_2300": (2300, (16, 16, 8), (2.0, 12.0), False, False),
    "crowded_6000": (6000, (200, 200, 16), (0.1, 0.6), False, False, (38.0, 38.0, 1.0, 42.0, 42.0, 5.0)),
}


@pytest.mark.parametrize("name", list(ROUTES))
def test_list_routes(name):
    from CudaGaussianVoxelizer import _C
    from oracle import g2v_oracle_c as OC
    n, dims, var, tiles_sorted, regions_sorted, *crowd = ROUTES[name]
    dev = torch.device("cuda")
    vr = (0.0, 0.0, 0.0) + tuple(0.4 * d + 0.1 for d in dims)
    w = W.Workload(name, n, 4, voxel_range=vr, var_range=var, extra={"mean_box": crowd[0]} if crowd else {})
    m, o, c, f = W.generate(w, seed=n)
    vs, vrn = np.array(w.voxel_size, np.float32), np.array(vr, np.float32)
    b = O.gaussian_boxes(m.numpy(), c.numpy(), vs, vrn)
    off, tid, gid, toff, sg = OC.csr(b["tile_lo"], b["tile_hi"], b["tiles"])
    print(f"[routes] {name} n={n} {dims} pairs={len(tid)}", flush=True)

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


# A batch's lists against those of its scenes alone, where the builds differ: the batch sorts (by the batch's tile
# ids and regions) what each scene lists; its offsets are scanned where each scene's workgroups sum them; and row
# lists of more than one scene.
#        scenes, n, voxels, variances, the batch sorts
BATCHES = {
    "sorted_2x1700": (2, 1700, (200, 200, 16), (0.1, 0.6), True),
    "scanned_2x300": (2, 300, (200, 200, 16), (0.5, 2.5), False),
    "row_lists_2x4200": (2, 4200, (40, 33, 16), (0.05, 0.2), False),
}


@pytest.mark.parametrize("name", list(BATCHES))
def test_batched_list_builds(name):
    from CudaGaussianVoxelizer import _C, PyCudaGaussianVoxelizer
    B, n, dims, var, sorts = BATCHES[name]
    dev = torch.device("cuda")
    vr = (0.0, 0.0, 0.0) + tuple(0.4 * d + 0.1 for d in dims)
    w = W.Workload(name, n, 4, voxel_range=vr, var_range=var, mean_pad=0.5)
    scenes = [[t.to(dev) for t in W.generate(w, seed=n + b)] for b in range(B)]
    vox = PyCudaGaussianVoxelizer(voxel_size=list(w.voxel_size), voxel_range=list(vr))
    g = torch.Generator(device=dev).manual_seed(2)
    gD = torch.randn(B, *dims, generator=g, device=dev)
    gF = torch.randn(B, *dims, 4, generator=g, device=dev)
    print(f"[batches] {name} {B} x {n} {dims}", flush=True)

    def step(leaves, *grads):
        leaves = [t.detach().clone().requires_grad_() for t in leaves]
        out = vox(*leaves)[:2]
        torch.autograd.backward(out, grads)
        return [t.detach() for t in out] + [t.grad for t in leaves]

    batch, ran = kernels(lambda: step([torch.stack(t) for t in zip(*scenes)], gD, gF))
    for kernel in ("k_fill_g2t", "k_fill_cells", "k_radix_scatter", "k_region_table"):
        assert (kernel in ran) == sorts, (kernel, ran)
    for b in range(B):
        alone, ran = kernels(lambda: step(scenes[b], gD[b], gF[b]))
        assert "k_radix_scatter" not in ran and "k_region_lists" in ran, ran
        for k, (x, y) in enumerate(zip(batch, alone)):
            assert torch.equal(x[b], y), (b, k)
    csr = _C._forward_batched(*[torch.stack(t) for t in zip(*scenes)][:3], w.voxel_size, vr,
                              torch.stack([s[3] for s in scenes]), keep_t2g=True)[3]["csr"]
    T = int(np.prod([-(-d // 4) for d in dims]))
    at = 0
    for b in range(B):
        one = _C._forward(*scenes[b][:3], w.voxel_size, vr, scenes[b][3], keep_t2g=True)[1]["csr"]
        M = one[0].numel()
        assert torch.equal(csr[0][at:at + M], one[0] + b * T) and torch.equal(csr[1][at:at + M], one[1] + b * n)
        assert torch.equal(csr[2][b * T:(b + 1) * T + 1], one[2] + at)
        at += M
    assert at == csr[0].numel()
