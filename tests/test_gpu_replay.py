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
    # (70 001 rays add into the leaves of a 64^3 grid in the order the GPU happens to take them: the bare difference of two such sums
    # is 5e-5 to 1.08e-4 from run to run, so large batches are held against the exact sum beyond the slack that any order has,
    # sqrt(terms) * 2^-24 * sum |term| of every element)
    ot = oracle_mod.Tree.from_n3tree(tree)
    want, slack = oracle_mod.volume_render_backward(ot, rays.origins, rays.dirs, rays.viewdirs, opt, go, n_threads=8, want_slack=True)
    err, ok = grad_close(got.cpu().numpy(), want, slack=slack if n > 1000 else None)
    assert ok, err
    target = torch.rand(n, 3, generator=gen).to(gpu)
    replayed, marched = C.se_grad(dev._spec(), rs, target, opt), C.se_grad(dev._spec(), rs, target, opt, workspace=False)
    assert torch.equal(replayed[0], marched[0])
    for a, b in zip(replayed[1:], marched[1:]):
        err, ok = grad_close(a.cpu().numpy(), b.cpu().numpy())
        assert ok, err


@pytest.mark.parametrize("levels,n,softplus", [(1, 160, False), (5, 1600, False), (5, 40007, True), (4, 40000, False), (5, 70001, False)])
@pytest.mark.parametrize("fmt", ["RGBA", "SH9"])
def test_notes_of_neighbours_that_share_leaves(gpu, oracle_mod, levels, n, softplus, fmt):
    """Pieces of 16 rays of which 1, 2, 3 ... 16 meet the scene, next to one another or (every fourth piece) from all
    over; their notes are read in slices of 64, 32, 16, 8 or 4 of each, up to 150 of them.

    The order slack of the oracle is taken off: up to 70 001 rays add into the leaves of a 32^3 or 64^3 grid in the order the
    GPU happens to take them, and the bare difference of two such sums is 4e-5 to 9.8e-5 from run to run.
    With softplus the generic kernels are the only reference: every leaf counts there, a leaf's density gradient is a
    difference of nearly equal sums, and the last bit of an exponential, which the device and the oracle round
    differently, is 1.9e-4 of the smallest of them, in the marching kernels' gradient bit for bit as in this one."""
    tree = svox.N3Tree(N=2, data_format=fmt, init_refine=levels)
    gen = torch.Generator().manual_seed(levels)
    tree.data.data.normal_(generator=gen)
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 0.5 * (torch.rand(tree.child.shape, generator=gen) < 0.8)
    rays = synth.sphere_rays(n, seed=n)
    at = torch.arange(n)
    piece, place = at // 16, at % 16
    near = piece % 4 != 3
    first = piece * 16
    dirs, origins = rays.dirs.clone(), rays.origins.clone()
    jitter = (torch.rand(n, 3, generator=gen) - 0.5) * 2e-3
    dirs[near] = torch.nn.functional.normalize(rays.dirs[first][near] + jitter[near], dim=-1)
    origins[near] = rays.origins[first][near]
    away = near & (place >= piece % 16 + 1)
    dirs[away] = -dirs[away]
    rays = svox.Rays(origins, dirs, dirs)
    opt = options(tree, step_size=1e-3, density_softplus=softplus)
    dev, rs = on_gpu(tree, gpu), rays_spec(rays, gpu)
    go = torch.randn(n, 3, generator=gen) * 1e-2
    out, notes = C.volume_render_noted(dev._spec(), rs, opt, records_per_ray=256)
    assert notes is not None
    got = C.volume_render_backward_noted(dev._spec(), rs, opt, go.to(gpu), notes)
    target = torch.rand(n, 3, generator=gen)
    replayed = C.se_grad(dev._spec(), rs, target.to(gpu), opt)
    marched = C.se_grad(dev._spec(), rs, target.to(gpu), opt, workspace=False)
    assert torch.equal(replayed[0], marched[0])
    if softplus:
        C.set_debug_flags(1)
        try:
            want = C.volume_render_backward(dev._spec(), rs, opt, go.to(gpu)).cpu().numpy()
        finally:
            C.set_debug_flags(0)
        checks = [(got, want, None)] + [(a, b.cpu().numpy(), None) for a, b in zip(replayed[1:], marched[1:])]
    else:
        ot = oracle_mod.Tree.from_n3tree(tree)
        ray_args = (ot, rays.origins, rays.dirs, rays.viewdirs)
        want, slack = oracle_mod.volume_render_backward(*ray_args, opt, go, n_threads=8, want_slack=True)
        _, g, h, g_slack, h_slack = oracle_mod.se_grad(*ray_args, target, opt, n_threads=8, want_slack=True)
        checks = [(got, want, slack), (replayed[1], g, g_slack), (replayed[2], h, h_slack)]
    for a, b, slack in checks:
        err, ok = grad_close(a.cpu().numpy(), b, slack=slack)
        assert ok, err


def test_notes_of_a_picture_taken_close_up(gpu):
    """Where neighbours share leaves their records are added together before they go to memory: the gradient of a
    picture taken from close to the tree is faster from notes than from a march of its own.  (A ray alone in its
    wavefront, whose records go out one by one, takes 5 780 us here, a march 4 360, rays with their neighbours 2 510.)"""
    tree = synth.dense_tree(6, data_format="SH16", seed=7, zero_fraction=0.5)
    dev = on_gpu(tree, gpu)
    opt = options(tree, step_size=1e-3)
    cam = C.CameraSpec()
    cam.c2w = synth.orbit_poses(1, seed=1, radius=1.2)[0][None].to(gpu)
    cam.width = cam.height = 800
    cam.fx = cam.fy = 1111.111
    go = torch.randn(1, 800, 800, 3, generator=torch.Generator().manual_seed(1)).to(gpu) * 1e-2
    spec = dev._spec()
    notes = C.volume_render_images_noted(spec, cam, opt, records_per_ray=256)[1]
    assert notes is not None
    times = {}
    for way in ["notes", "march"] * 6:
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        if way == "notes":
            C.volume_render_images_backward_noted(spec, cam, opt, go, notes)
        else:
            C.volume_render_images_backward(spec, cam, opt, go, workspace=False)
        end.record()
        end.synchronize()
        times.setdefault(way, []).append(begin.elapsed_time(end) * 1e3)
    noted, marched = (sorted(times[w])[3] for w in ("notes", "march"))
    print(f"[notes] close up: from notes {noted:.0f} us, from a march {marched:.0f} us", flush=True)
    assert noted <= 0.9 * marched


@pytest.mark.parametrize("fmt,softplus,density", [("SH4", False, 2000.0), ("RGBA", False, 1e4), ("SH9", False, 1e36), ("SH1", True, 300.0)])
@pytest.mark.parametrize("flags", [0, 2, 4, 8])
def test_noted_rays_end_where_nothing_shines_through(gpu, oracle_mod, fmt, softplus, density, flags):
    """Leaves so dense that a ray's transmittance falls below the smallest float inside the tree: its notes end there, picture and
    gradients stay those of the whole ray.  Where the picture shades none of them, none are left out."""
    n = 700
    tree = svox.N3Tree(N=2, data_format=fmt, init_refine=4)
    gen = torch.Generator().manual_seed(11)
    tree.data.data.normal_(generator=gen)
    dense = torch.rand(tree.child.shape, generator=gen)
    tree.data.data[..., -1] = torch.where(dense < 0.5, density * dense, -3.0 * dense)
    rays = synth.sphere_rays(n, seed=12)
    dev, rs = on_gpu(tree, gpu), rays_spec(rays, gpu)
    spec, ot = dev._spec(), oracle_mod.Tree.from_n3tree(tree)
    go, target = torch.randn(n, 3, generator=gen) * 1e-2, torch.full((n, 3), 0.5, device=gpu)
    for thresh in (0.0, float("inf")):
        opt = options(tree, step_size=1e-3, density_softplus=softplus, sigma_thresh=thresh, stop_thresh=0.0)
        positive = C.volume_render_stats(spec, rs, opt)["samples_bwd_pos"]
        C.set_debug_flags(flags)
        try:
            out, notes = C.volume_render_noted(spec, rs, opt, records_per_ray=256)
            got = C.volume_render_backward_noted(spec, rs, opt, go.to(gpu), notes)
            alone = C.volume_render_backward(spec, rs, opt, go.to(gpu))
            colours = C.se_grad(spec, rs, target, opt)[0]
        finally:
            C.set_debug_flags(0)
        noted = notes.view(torch.int32)[: n * 96].view(n, 96)[:, 91]      # (how many notes a ray has: beside the link of its first chunk)
        assert bool((noted >= 0).all())
        assert int(noted.sum()) == positive if thresh > 0 else int(noted.sum()) < 0.9 * positive
        # (with softplus the last bit of its exponential differs between device and oracle: the marching kernels are the reference)
        C.set_debug_flags(1 if softplus else 0)
        try:
            march, march_se = C.volume_render(spec, rs, opt), C.se_grad(spec, rs, target, opt, workspace=False)[0]
            march_grad = C.volume_render_backward(spec, rs, opt, go.to(gpu), workspace=False).cpu().numpy()
        finally:
            C.set_debug_flags(0)
        if not softplus:
            assert (out.cpu().numpy() == oracle_mod.volume_render(ot, rays.origins, rays.dirs, rays.viewdirs, opt)).all()
            march_grad = oracle_mod.volume_render_backward(ot, rays.origins, rays.dirs, rays.viewdirs, opt, go)
        assert torch.equal(out, march) and torch.equal(colours, march_se)
        for what, grad in (("from notes", got), ("alone", alone)):
            err, ok = grad_close(grad.cpu().numpy(), march_grad, what=what)
            assert ok, (thresh, what, err)
