"""Double-precision octrees on the kernels that give four lanes to a ray (group_kernels.h).

Bar: forward renders bit-identical to the oracle and to the one-ray-per-lane kernels; gradients within 1e-4 of the
oracle's exact sum and 1e-9 of the one-ray-per-lane kernels'.
"""
import numpy as np
import pytest
import torch

import svox_amd as svox
from svox_amd import csrc as C
from svox_amd import synth
from util import cam_spec, grad_close, on_gpu, options, rays_spec

pytestmark = pytest.mark.gpu


def both_kernels(fn):
    """fn() on the kernels of group_kernels.h and on the one-ray-per-lane kernels"""
    got = fn()
    C.set_debug_flags(1)
    try:
        return got, fn()
    finally:
        C.set_debug_flags(0)


@pytest.mark.parametrize("fmt,n,kw", [("RGBA", 1000 + 13, {}), ("SH1", 15, {}), ("SH4", 1, {}), ("SH9", 1000 + 13, {"fast": True}),
                                      ("SH16", 700, {"density_softplus": True, "rgb_padding": 0.001}), ("SH25", 333, {}),
                                      ("SH9", 500, {"min_comp": 1, "max_comp": 3}), ("SG4", 500, {}),
                                      # (more leaves with density along a ray than the gradient's list holds)
                                      ("SH4 dense", 300, {})])
def test_rays_and_gradients(gpu, oracle_mod, fmt, n, kw):
    tree = synth.shell_tree(depth=5, n_spheres=5, data_format="SH4" if fmt in ("SG4", "SH4 dense") else fmt, seed=7, sigma_range=(2.0, 40.0)).double()
    if fmt == "SH4 dense":
        tree = svox.N3Tree(N=2, data_format="SH4", init_refine=5, dtype=torch.float64)
        tree.data.data.normal_(generator=torch.Generator().manual_seed(6))
        tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 0.3 + 0.01
    if fmt == "SG4":
        tree.data_format = svox.DataFormat("SG4")
        tree.extra_data = torch.cat([torch.rand(4, 1, dtype=torch.float64) * 4 + 0.5,
                                     synth.unit_vectors(4, torch.Generator().manual_seed(3)).double()], dim=1)
    rays = synth.sphere_rays(n, seed=4, dtype=torch.float64)
    opt = options(tree, step_size=1e-3, **kw)
    dev, rs = on_gpu(tree, gpu), rays_spec(rays, gpu)
    if fmt == "SG4":
        dev.extra_data = tree.extra_data.to(gpu)
    out, generic = both_kernels(lambda: C.volume_render(dev._spec(), rs, opt))
    assert torch.equal(out, generic)
    ot = oracle_mod.Tree.from_n3tree(tree)
    if not kw.get("density_softplus"):      # (its logarithm is the platform's)
        assert np.array_equal(out.cpu().numpy(), oracle_mod.volume_render(ot, rays.origins, rays.dirs, rays.viewdirs, opt))
    go = torch.randn(n, 3, generator=torch.Generator().manual_seed(5), dtype=torch.float64) * 1e-2
    grad, generic = both_kernels(lambda: C.volume_render_backward(dev._spec(), rs, opt, go.to(gpu)))
    assert (grad - generic).abs().max() <= 1e-9 * generic.abs().max()
    want = oracle_mod.volume_render_backward(ot, rays.origins, rays.dirs, rays.viewdirs, opt, go)
    err, ok = grad_close(grad.cpu().numpy(), want)
    assert ok, err


def test_pictures_and_trees_deeper_than_the_integer_coordinates(gpu, oracle_mod):
    tree, point = synth.deep_tree(27, "SH4", seed=5, dtype=torch.float64)
    gen = torch.Generator().manual_seed(2)
    origins = 0.5 + 1.5 * synth.unit_vectors(200, gen).double()
    dirs = point - origins                                       # all of them through the deepest leaf
    dirs = dirs / dirs.norm(dim=-1, keepdim=True)
    rays = svox.Rays(origins.contiguous(), dirs.contiguous(), dirs.clone())
    opt = options(tree, step_size=1e-4)
    dev = on_gpu(tree, gpu)
    out, generic = both_kernels(lambda: C.volume_render(dev._spec(), rays_spec(rays, gpu), opt))
    assert torch.equal(out, generic)
    tree = synth.shell_tree(depth=5, n_spheres=5, data_format="SH4", seed=7, sigma_range=(2.0, 40.0)).double()
    dev = on_gpu(tree, gpu)
    cam = cam_spec(synth.orbit_poses(1, seed=4, radius=2.5)[0], 37, 29, 40.0, device=gpu, dtype=torch.float64)
    for opt in (options(tree, step_size=1e-3), options(tree, step_size=1e-3, ndc=svox.NDCConfig(37, 29, 40.0), fast=True)):
        out, generic = both_kernels(lambda: C.volume_render_image(dev._spec(), cam, opt))
        assert torch.equal(out, generic)
        go = torch.randn(29, 37, 3, generator=gen, dtype=torch.float64).to(gpu)
        grad, generic = both_kernels(lambda: C.volume_render_image_backward(dev._spec(), cam, opt, go))
        assert (grad - generic).abs().max() <= 1e-9 * generic.abs().max()


@pytest.mark.parametrize("flags", [2, 4, 32])
@pytest.mark.parametrize("fmt,kw", [("RGBA", {}), ("SH9", {"fast": True}), ("SH4", {"density_softplus": True, "min_comp": 1, "max_comp": 2})])
def test_rays_walked_by_four_lanes_together(gpu, flags, fmt, kw):
    """Any debug flag but those for pieces takes the kernels whose four lanes share a walk, for few rays too: lists of leaves that run over
    (every leaf of 64^3 has density) and a number of rays that is no multiple of a wavefront's."""
    n = 333
    gen = torch.Generator().manual_seed(3)
    tree = svox.N3Tree(N=2, data_format=fmt, init_refine=5, dtype=torch.float64)
    tree.data.data.normal_(generator=gen)
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 0.3 + 0.01
    rays = synth.sphere_rays(n, seed=4, dtype=torch.float64)
    rays.dirs[::5] *= -1.0
    opt = options(tree, step_size=1e-3, **kw)
    spec, rs = on_gpu(tree, gpu)._spec(), rays_spec(rays, gpu)
    go = torch.randn(n, 3, generator=gen, dtype=torch.float64).to(gpu)

    def passes(f):
        C.set_debug_flags(f)
        try:
            return C.volume_render(spec, rs, opt), C.volume_render_backward(spec, rs, opt, go)
        finally:
            C.set_debug_flags(0)

    (out, grad), (want, ref) = passes(flags), passes(1)
    assert torch.equal(out, want)
    assert (grad - ref).abs().max() <= 1e-11 * ref.abs().max()
