"""Gradients from notes at the edges of the replay kernels: chunks of 15 notes, batches of 64 lanes and 32 rays, rays
with more than 64 notes, more chunks than a block keeps track of, blocks of 16, 32 and 64 rays.

Bar: gradients within 1e-4 of the oracle's exact sum (small batches) or of the generic kernels' (large ones); the
colours of se_grad bit-identical to the marching kernel's.
"""
import pytest
import torch

import svox_amd as svox
from svox_amd import csrc as C
from svox_amd import synth
from util import grad_close, on_gpu, options, rays_spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels,keep,n", [(0, 1.0, 33), (2, 0.2, 1000), (3, 1.0, 15), (4, 0.3, 17), (5, 1.0, 300), (5, 0.6, 40000), (5, 1.0, 70001)])
@pytest.mark.parametrize("fmt", ["SH1", "SH9"])
def test_notes_of_every_number(gpu, oracle_mod, levels, keep, n, fmt):
    tree = svox.N3Tree(N=2, data_format=fmt, init_refine=levels)
    gen = torch.Generator().manual_seed(levels)
    tree.data.data.normal_(generator=gen)
    # (thin enough for the far end of a ray to count)
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 0.5 * (torch.rand(tree.child.shape, generator=gen) < keep)
    rays = synth.sphere_rays(n, seed=n)
    opt = options(tree, step_size=1e-3)
    dev, rs = on_gpu(tree, gpu), rays_spec(rays, gpu)
    go = torch.randn(n, 3, generator=gen) * 1e-2
    out, notes = C.volume_render_noted(dev._spec(), rs, opt, records_per_ray=256)
    assert notes is not None
    got = C.volume_render_backward_noted(dev._spec(), rs, opt, go.to(gpu), notes)
    if n <= 1000:
        ot = oracle_mod.Tree.from_n3tree(tree)
        want = oracle_mod.volume_render_backward(ot, rays.origins, rays.dirs, rays.viewdirs, opt, go)
    else:
        C.set_debug_flags(1)
        try:
            want = C.volume_render_backward(dev._spec(), rs, opt, go.to(gpu)).cpu().numpy()
        finally:
            C.set_debug_flags(0)
    err, ok = grad_close(got.cpu().numpy(), want)
    assert ok, err
    target = torch.rand(n, 3, generator=gen).to(gpu)
    replayed, marched = C.se_grad(dev._spec(), rs, target, opt), C.se_grad(dev._spec(), rs, target, opt, workspace=False)
    assert torch.equal(replayed[0], marched[0])
    for a, b in zip(replayed[1:], marched[1:]):
        err, ok = grad_close(a.cpu().numpy(), b.cpu().numpy())
        assert ok, err
