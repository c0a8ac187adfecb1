"""Gradients whose arrays are cleared by the launch that takes the notes: on memory that held NaN, in every shape of that launch, for sizes
that are no multiple of a block's share or of 16 bytes.

Bar: the arrays are those of the same call without a workspace, which clears them by themselves -- within 1e-4 beyond the order slack of
the sums, and not a number of the memory before left in them.  Which leaves no ray has anything for, the Hessian diagonal says: a sum of squares
is 0 where all of its terms are and nowhere else, in whatever order they are added, while the terms of a gradient may cancel to exactly 0 in one order
and not in another.
"""
import pytest
import torch

import svox_amd as svox
from svox_amd import csrc as C
from svox_amd import synth
from util import cam_spec, grad_close, on_gpu, options, rays_spec

pytestmark = pytest.mark.gpu


def dirty(like, gpu):
    """leaves NaN where the next arrays of that size will lie"""
    for t in [torch.full((like,), float("nan"), device=gpu) for _ in range(3)]:
        del t


def untouched(hessian):
    return (hessian == 0).all(-1)


def check_untouched(got, nobodys, hessian, what):
    """every element of the leaves `nobodys` is 0"""
    stray = (got != 0) & nobodys[..., None]
    if bool(stray.any()):
        at = stray.nonzero()
        lines = [f"{tuple(i.tolist())}: {float(got[tuple(i)])!r}, Hessian {float(hessian[tuple(i)])!r}" for i in at[:8]]
        pytest.fail(f"{what}: {len(at)} elements of leaves that no ray has anything for are not 0: " + "; ".join(lines), pytrace=False)


@pytest.mark.parametrize("flags", [0, 2, 4, 8, 32 | 62 << 8, 64 | 255 << 8, 64 | 16 << 16, 64 | 2])
@pytest.mark.parametrize("N,levels,fmt", [(2, 4, "SH9"), (3, 2, "SH1"), (3, 0, "RGBA"), (2, 5, "SH4")])
def test_cleared_by_the_noting_launch(gpu, flags, N, levels, fmt):
    n = 400
    gen = torch.Generator().manual_seed(levels)
    tree = svox.N3Tree(N=N, data_format=fmt, init_refine=levels)
    tree.data.data.normal_(generator=gen)
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() * (torch.rand(tree.child.shape, generator=gen) < 0.2)
    dev, rs = on_gpu(tree, gpu), rays_spec(synth.sphere_rays(n, seed=3), gpu)
    spec, opt = dev._spec(), options(tree, step_size=1e-3)
    go, target = (torch.randn(n, 3, generator=gen) * 1e-2).to(gpu), torch.rand(n, 3, generator=gen).to(gpu)
    cam = cam_spec(synth.orbit_poses(1, seed=2, radius=3.0)[0], 21, 19, 30.0, device=gpu)
    go_image, image = go[:399].reshape(19, 21, 3).contiguous(), target[:399].reshape(19, 21, 3).contiguous()
    calls = [lambda ws: C.volume_render_backward(spec, rs, opt, go, workspace=ws), lambda ws: C.se_grad(spec, rs, target, opt, workspace=ws),
             lambda ws: C.volume_render_image_backward(spec, cam, opt, go_image, workspace=ws),
             lambda ws: C.se_grad_persp(spec, cam, opt, image, workspace=ws)]
    hessians = [calls[k](False)[2] for k in (1, 3)]
    for k, call in enumerate(calls):
        want = call(False)
        dirty(tree.data.numel(), gpu)
        C.set_debug_flags(flags)
        try:
            got = call(True)
        finally:
            C.set_debug_flags(0)
        pairs = zip(got, want) if isinstance(got, (tuple, list)) else [(got, want)]
        for a, b in pairs:
            assert bool(torch.isfinite(a).all()), k
            # (at most 400 terms of a leaf, added in another order: 20 * 2^-24 of the sum of their sizes on each side)
            err, ok = grad_close(a.cpu().numpy(), b.cpu().numpy(), what=f"call {k}")
            assert ok, (k, err)
            if a.shape == tree.data.shape:
                check_untouched(a, untouched(hessians[k // 2]), hessians[k // 2], f"call {k}")


@pytest.mark.parametrize("n", [32768, 32769])
def test_much_to_clear_beside_many_rays(gpu, n):
    """Arrays of 1.2 GB each, on either side of the number of rays from which on they are cleared before the march."""
    tree = synth.shell_tree(depth=9, data_format="SH16", n_spheres=24, seed=0, device=gpu)
    rs, opt, spec = rays_spec(synth.sphere_rays(n, seed=5), gpu), options(tree, step_size=5e-4), tree._spec()
    target = torch.rand(n, 3, generator=torch.Generator().manual_seed(n)).to(gpu)
    dirty(tree.data.numel(), gpu)
    got, want = C.se_grad(spec, rs, target, opt), C.se_grad(spec, rs, target, opt, workspace=False)
    assert torch.equal(got[0], want[0])
    nobodys = untouched(want[2])
    assert torch.equal(untouched(got[2]), nobodys)
    for what, a in zip(("gradient", "Hessian"), got[1:]):
        assert bool(torch.isfinite(a).all())
        check_untouched(a, nobodys, want[2], what)
