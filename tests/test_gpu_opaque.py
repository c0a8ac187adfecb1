"""What lies behind leaves that let next to nothing through, and numbers that are none, in the passes that take notes, walk rays in
pieces or list them.

Bar: pictures equal bit for bit to those of the kernels that march a ray from end to end (NaN where they have one); gradients finite
where theirs are, the terms of one leaf within 1e-4 of theirs (sums of a few terms in another order).
"""
import pytest
import torch

import svox_amd as svox
from svox_amd import csrc as C
from svox_amd import synth
from util import grad_close, on_gpu, options, rays_spec

pytestmark = pytest.mark.gpu

PIECES, LISTED = 32 | 62 << 8, 64 | 16 << 16
FLAGS = [0, 2, 4, 8, PIECES, LISTED]


def run(flags, f):
    C.set_debug_flags(flags)
    try:
        return f()
    finally:
        C.set_debug_flags(0)


def same(a, b):
    return bool(((a == b) | (a.isnan() & b.isnan())).all())


def layers(depths, fmt="SH4", seed=3):
    """A 16^3 grid whose layers along z have these optical depths (empty beyond), rays along z through it, and where the leaves of a
    layer are in tree.data."""
    tree = svox.N3Tree(N=2, data_format=fmt, init_refine=3)
    gen = torch.Generator().manual_seed(seed)
    tree.data.data.normal_(generator=gen)
    tree.data.data[..., -1] = 0.0
    leaves = (tree.child == 0).nonzero()
    layer = (synth._leaf_corners(tree, leaves)[:, 2] * 16).round().long()
    at = [tuple(leaves[layer == k].T) for k in range(len(depths))]
    for k, depth in enumerate(depths):
        tree.data.data[at[k] + (-1,)] = depth / (1 / 16 + 1e-3)
    n = 500
    origins = torch.rand(n, 3, generator=gen)
    origins[:, 2] = -1.0
    dirs = torch.tensor([[0.0, 0.0, 1.0]]).expand(n, 3).contiguous()
    return tree, svox.Rays(origins, dirs, synth.unit_vectors(n, gen)), at, gen


@pytest.mark.parametrize("flags", FLAGS)
@pytest.mark.parametrize("stop_thresh", [0.0, -1.0, 1e-3])
@pytest.mark.parametrize("hidden", ["nan", "finite"])
def test_noted_pictures_behind_dense_layers(gpu, flags, stop_thresh, hidden):
    """A transmittance of e^-92 -- below the smallest normal float, above the smallest one -- in front of leaves with NaN coefficients, and
    of a background that such a factor brings back into the range: a picture that takes notes is the picture that does not."""
    tree, rays, at, _ = layers([46.0, 46.0, 0.3])
    if hidden == "nan":
        tree.data.data[at[2] + (slice(0, -1),)] = float("nan")
    spec, rs = on_gpu(tree, gpu)._spec(), rays_spec(rays, gpu)
    for bg in (1.0, 1e38):
        opt = options(tree, step_size=1e-3, stop_thresh=stop_thresh, background_brightness=bg)
        want = run(1, lambda: C.volume_render(spec, rs, opt))
        assert bool(want.isnan().all()) == (hidden == "nan" and stop_thresh <= 0.0)
        out, notes = run(flags, lambda: C.volume_render_noted(spec, rs, opt, records_per_ray=64))
        assert notes is not None and same(out, want)
        assert same(run(flags, lambda: C.volume_render(spec, rs, opt)), want)
        if stop_thresh == 0.0:
            target = torch.rand(want.shape, generator=torch.Generator().manual_seed(1)).to(gpu)
            marched = run(1, lambda: C.se_grad(spec, rs, target, opt, workspace=False))[0]
            assert same(run(flags, lambda: C.se_grad(spec, rs, target, opt))[0], marched)


@pytest.mark.parametrize("flags", FLAGS)
def test_gradients_of_what_shines_through_faintly_scale(gpu, flags):
    """The gradient of the picture scaled by 1e35: the colour gradients of leaves behind e^-92 are numbers of ordinary size."""
    tree, rays, at, gen = layers([46.0, 46.0, 0.3])
    spec, rs = on_gpu(tree, gpu)._spec(), rays_spec(rays, gpu)
    opt = options(tree, step_size=1e-3)
    go = (torch.randn(rays.origins.shape, generator=gen) * 1e35).to(gpu)
    want = run(1, lambda: C.volume_render_backward(spec, rs, opt, go, workspace=False))

    def from_notes():
        notes = C.volume_render_noted(spec, rs, opt, records_per_ray=64)[1]
        return C.volume_render_backward_noted(spec, rs, opt, go, notes)

    hidden = at[2] + (slice(0, -1),)
    assert want[hidden].abs().max() > 1e-7
    for got in (run(flags, from_notes), run(flags, lambda: C.volume_render_backward(spec, rs, opt, go))):
        err, ok = grad_close(got[hidden].cpu().numpy(), want[hidden].cpu().numpy())
        assert ok, err


@pytest.mark.parametrize("flags", FLAGS)
def test_gradients_end_where_the_transmittance_is_zero(gpu, flags):
    """Behind e^-120 no finite coefficient counts; one that is NaN, and not in the next few leaves, reaches the gradient of passes without
    notes only."""
    tree, rays, at, gen = layers([60.0, 60.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.3])
    opt = options(tree, step_size=1e-3)
    rs, go = rays_spec(rays, gpu), torch.randn(rays.origins.shape, generator=gen).to(gpu)
    want = run(1, lambda: C.volume_render_backward(on_gpu(tree, gpu)._spec(), rs, opt, go, workspace=False))
    assert bool((want[at[7] + (slice(0, -1),)] == 0).all())
    tree.data.data[at[7] + (slice(0, -1),)] = float("nan")
    spec = on_gpu(tree, gpu)._spec()
    assert bool(run(1, lambda: C.volume_render_backward(spec, rs, opt, go, workspace=False)).isnan().any())

    def from_notes():
        out, notes = C.volume_render_noted(spec, rs, opt, records_per_ray=64)
        assert same(out, C.volume_render(spec, rs, opt))
        return C.volume_render_backward_noted(spec, rs, opt, go, notes)

    for got in (run(flags, from_notes), run(flags, lambda: C.volume_render_backward(spec, rs, opt, go))):
        for k in (0, 1):
            err, ok = grad_close(got[at[k]].cpu().numpy(), want[at[k]].cpu().numpy())
            assert ok, (k, err)
        assert bool((got[at[7]] == 0).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("kind", ["grid", "shell"])
def test_values_that_are_no_numbers(gpu, dtype, kind):
    """NaN, infinite and extreme coefficients and densities all over a tree: every way through it gives the pictures of the kernels with
    one ray per lane.  Without densities that end a ray, gradients are finite where theirs are, and close to them."""
    n = 700
    gen = torch.Generator().manual_seed(5)
    tree = svox.N3Tree(N=2, data_format="SH4", init_refine=4) if kind == "grid" else synth.shell_tree(depth=6, data_format="SH4", n_spheres=6, seed=4)
    tree.data.data[..., :-1].normal_(generator=gen)
    tree.data.data[..., -1] = 4.0 * torch.rand(tree.child.shape, generator=gen) * (torch.rand(tree.child.shape, generator=gen) < 0.5)
    odd = torch.rand(tree.data.shape, generator=gen)
    inf, most = float("inf"), torch.finfo(torch.float32).max
    for k, v in enumerate((float("nan"), inf, -inf, most, -most)):
        tree.data.data[..., :-1][(odd[..., :-1] * 2000).long() == k] = v
    for k, v in enumerate((float("nan"), -inf, -most, -1.0)):
        tree.data.data[..., -1][(odd[..., -1] * 300).long() == k] = v
    rays = synth.sphere_rays(n, seed=6, dtype=dtype)
    rs = rays_spec(rays, gpu)
    go = (torch.randn(n, 3, generator=gen, dtype=dtype) * 1e-2).to(gpu)
    flags = FLAGS if dtype == torch.float32 else [0, 32 | 216 << 8, 32 | 601 << 8]
    for dense in (False, True):
        if dense:
            for k, v in enumerate((inf, most, 1e4)):
                tree.data.data[..., -1][(odd[..., -1] * 300).long() == 10 + k] = v
        spec = on_gpu(tree.to(dtype), gpu)._spec()
        for kw in ({}, {"density_softplus": True}, {"sigma_thresh": 1.0, "stop_thresh": 0.3}):
            opt = options(tree, step_size=1e-3, **kw)
            want = run(1, lambda: C.volume_render(spec, rs, opt))
            grad = run(1, lambda: C.volume_render_backward(spec, rs, opt, go, workspace=False))
            assert bool(want.isnan().any()) and not bool(want.isnan().all())
            for f in flags:
                assert same(run(f, lambda: C.volume_render(spec, rs, opt)), want), (kw, f)
                if dtype == torch.float32:
                    out, notes = run(f, lambda: C.volume_render_noted(spec, rs, opt, records_per_ray=256))
                    assert same(out, want), (kw, f)
                if dense and dtype == torch.float32:
                    continue
                got = [run(f, lambda: C.volume_render_backward(spec, rs, opt, go))]
                if dtype == torch.float32:
                    got.append(run(f, lambda: C.volume_render_backward_noted(spec, rs, opt, go, notes)))
                for g in got:
                    assert torch.equal(g.isfinite(), grad.isfinite()), (kw, f)
                    fine = grad.isfinite()
                    err, ok = grad_close(g[fine].cpu().numpy(), grad[fine].cpu().numpy())
                    assert ok, (kw, f, err)


@pytest.mark.parametrize("flags", FLAGS)
@pytest.mark.parametrize("N", [2, 3])
def test_directions_without_a_length(gpu, oracle_mod, flags, N):
    """The norm of a tiny direction is zero and its unit vector infinite: from an infinite origin the first sample has no number for a coordinate, and
    counts as the upper corner.  (Every leaf ends such a ray.)"""
    inf, tiny = float("inf"), 1e-30
    signs = torch.tensor([[x, y, z] for x in (1, -1) for y in (1, -1) for z in (1, -1)], dtype=torch.float32)
    origins = torch.cat([signs * inf] * 3 + [torch.rand(8, 3, generator=torch.Generator().manual_seed(2))])
    dirs = torch.cat([signs * tiny, -signs * tiny, signs * 0.0, signs * tiny])
    gen = torch.Generator().manual_seed(1)
    tree = svox.N3Tree(N=N, data_format="SH1", init_refine=1)
    tree.data.data.normal_(generator=gen)
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() + 1.0
    rays = svox.Rays(origins, dirs, synth.unit_vectors(32, gen))
    spec, rs, opt = on_gpu(tree, gpu)._spec(), rays_spec(rays, gpu), options(tree, step_size=1e-3)
    want = torch.from_numpy(oracle_mod.volume_render(oracle_mod.Tree.from_n3tree(tree), rays.origins, rays.dirs, rays.viewdirs, opt))
    assert torch.equal(run(1, lambda: C.volume_render(spec, rs, opt)).cpu(), want)
    assert torch.equal(run(flags, lambda: C.volume_render(spec, rs, opt)).cpu(), want)
    assert torch.equal(run(flags, lambda: C.volume_render_noted(spec, rs, opt)[0]).cpu(), want)
