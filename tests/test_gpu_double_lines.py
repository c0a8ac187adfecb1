"""Double precision on either side of the lines between rays in pieces and lanes that walk a ray together, and lists that run over, after which
a piece's walk starts at the root again (render_group_kernel): the kernels with one ray per lane are the reference."""
import pytest
import torch

import svox_amd as svox
from svox_amd import csrc as C
from svox_amd import synth
from util import options, rays_spec

pytestmark = pytest.mark.gpu


def run(flags, fn):
    C.set_debug_flags(flags)
    try:
        return fn()
    finally:
        C.set_debug_flags(0)


# (levels, rays, rays to a wavefront and log2 of their pieces, or None: the rule)
@pytest.mark.parametrize("levels,n,split", [(3, 32769, None), (3, 65536, None), (3, 65537, None), (5, 26624, None), (5, 26625, None), (5, 28673, None),
                                            (6, 40961, None), (6, 65537, None), (6, 300, (16, 2)), (6, 300, (12, 2)), (7, 300, (8, 3))])
def test_lines_and_lists_that_run_over(gpu, levels, n, split):
    gen = torch.Generator(device=gpu).manual_seed(levels)
    tree = svox.N3Tree(N=2, data_format="SH1", init_refine=levels, device=gpu, dtype=torch.float64)
    tree.data.data.normal_(generator=gen)
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 0.1 + 0.01
    rs, opt, spec = rays_spec(synth.sphere_rays(n, seed=5, dtype=torch.float64), gpu), options(tree, step_size=1e-3), tree._spec()
    go = torch.randn(n, 3, generator=gen, device=gpu, dtype=torch.float64)

    def passes():
        return C.volume_render(spec, rs, opt), C.volume_render_backward(spec, rs, opt, go)

    want = run(1, passes)
    got = run(0 if split is None else 32 | (split[0] + 100 * split[1]) << 8, passes)
    assert torch.equal(got[0], want[0])
    # (up to n terms of a leaf in another order: n * 2^-53 of the sum of their sizes at most, which cancels to a hundredth of it)
    assert (got[1] - want[1]).abs().max() <= n * 1.2e-14 * want[1].abs().max()


@pytest.mark.parametrize("levels,fmt", [(3, "RGBA"), (3, "SH9"), (4, "SH4"), (4, "SH9")])
@pytest.mark.parametrize("size", [128, 144, 160, 176])
def test_pictures_on_either_side(gpu, levels, fmt, size):
    """Small trees have gradients of pictures in pieces up to 20 480 pixels, those of 32^3 leaves pictures of few functions up to as many and others up to 26 624."""
    gen = torch.Generator(device=gpu).manual_seed(levels)
    tree = svox.N3Tree(N=2, data_format=fmt, init_refine=levels, device=gpu, dtype=torch.float64)
    tree.data.data.normal_(generator=gen)
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 0.1 + 0.01
    opt, spec, cam = options(tree, step_size=1e-3), tree._spec(), C.CameraSpec()
    cam.c2w = synth.orbit_poses(1, seed=3, radius=2.5)[0].to(gpu).double().contiguous()
    cam.fx, cam.fy, cam.width, cam.height = size * 1.4, size * 1.4, size, size
    go = torch.randn(size, size, 3, generator=gen, device=gpu, dtype=torch.float64)

    def passes():
        return C.volume_render_image(spec, cam, opt), C.volume_render_image_backward(spec, cam, opt, go)

    want, got = run(1, passes), run(0, passes)
    assert torch.equal(got[0], want[0])
    # (as above)
    assert (got[1] - want[1]).abs().max() <= size * size * 1.2e-14 * want[1].abs().max()
