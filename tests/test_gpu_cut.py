"""Rays walked in pieces, several lanes to a ray: every split of a wavefront (one to eight rays, one to 64 pieces), lists that run over,
rays that miss, end early, or whose notes find no room.

Bar: pictures and noted colours bit-identical to those of the kernel that walks a ray from end to end, as many notes of every
ray, gradients within 1e-4 of that kernel's -- the terms are the same, added in another order -- beyond the order slack where the
oracle has one.
"""
import pytest
import torch

import svox_amd as svox
from svox_amd import csrc as C
from svox_amd import synth
from util import cam_spec, grad_close, on_gpu, options, rays_spec

pytestmark = pytest.mark.gpu

END_TO_END = 4


def cut(per_wave, most):
    return 32 | (per_wave + 10 * most) << 8


def run(flags, f):
    C.set_debug_flags(flags)
    try:
        return f()
    finally:
        C.set_debug_flags(0)


def scene(kind, fmt, gen):
    if kind == "shell":
        return synth.shell_tree(depth=7, data_format=fmt, n_spheres=6, seed=4)
    if kind == "deep":
        return synth.deep_tree(12, data_format=fmt, seed=5)[0]
    extra = torch.randn(4, 4, generator=gen) if fmt.startswith("SG") else None
    tree = svox.N3Tree(N=3 if kind == "thirds" else 2, data_format=fmt, init_refine={"thirds": 2, "leaf": 0, "dense": 5}[kind], extra_data=extra)
    tree.data.data.normal_(generator=gen)
    keep = torch.rand(tree.child.shape, generator=gen) < 0.6
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 3 * keep
    return tree


@pytest.mark.parametrize("per_wave,most", [(8, 0), (8, 6), (5, 2), (3, 6), (2, 5), (1, 6)])
@pytest.mark.parametrize("kind,fmt,softplus,fast", [("dense", "SH9", False, False), ("dense", "RGBA", True, False), ("thirds", "SG4", False, False),
                                                    ("shell", "SH16", False, True), ("deep", "SH4", False, False), ("leaf", "SH25", False, True)])
def test_rays_in_pieces_are_the_rays_from_end_to_end(gpu, oracle_mod, monkeypatch, kind, fmt, softplus, fast, per_wave, most):
    n = 301
    gen = torch.Generator().manual_seed(7)
    tree = scene(kind, fmt, gen)
    rays = synth.sphere_rays(n, seed=8)
    rays.dirs[::7] *= -1.0                              # (some look away)
    rays.dirs[5] = torch.tensor([0.0, 0.0, 1.0])        # (and one along an axis)
    opt = options(tree, step_size=1e-3, density_softplus=softplus, fast=fast)
    dev, rs = on_gpu(tree, gpu), rays_spec(rays, gpu)
    go, target = (torch.randn(n, 3, generator=gen) * 1e-2).to(gpu), torch.rand(n, 3, generator=gen).to(gpu)
    plain, marked = dev._spec(), dev._spec()
    marked.child_marks = C.mark_empty_leaves(plain, density_softplus=softplus)
    marked.child_marks_softplus = softplus
    slack = None
    if not softplus:
        ot = oracle_mod.Tree.from_n3tree(tree)
        slack = oracle_mod.volume_render_backward(ot, rays.origins, rays.dirs, rays.viewdirs, opt, go.cpu(), want_slack=True)[1]

    def passes(spec):
        out, notes = C.volume_render_noted(spec, rs, opt, records_per_ray=256)
        count = notes.view(torch.int32)[: n * 96].view(n, 96)[:, 91].clone()
        return (C.volume_render(spec, rs, opt), out, count, C.se_grad(spec, rs, target, opt)[0],
                C.volume_render_backward_noted(spec, rs, opt, go, notes), C.volume_render_backward(spec, rs, opt, go))

    for spec in (plain, marked):
        want, got = run(END_TO_END, lambda: passes(spec)), run(cut(per_wave, most), lambda: passes(spec))
        for what, a, b in zip(("picture", "noted picture", "notes", "colours"), got, want):
            assert torch.equal(a, b), what
        for what, a, b in zip(("from notes", "alone"), got[4:], want[4:]):
            err, ok = grad_close(a.cpu().numpy(), b.cpu().numpy(), slack=slack, what=what)
            assert ok, (what, err)
    # room for as many chunks of 15 notes as the rays need, beside the first of each: none are lost
    monkeypatch.setattr(C, "SMALL_BATCH_ROOM", 1)
    chunks = -(-int(((want[2] - 1).clamp(min=0) // 15).sum()) // n) + 1
    notes = run(cut(per_wave, most), lambda: C.volume_render_noted(plain, rs, opt, records_per_ray=15 * chunks))[1]
    assert torch.equal(notes.view(torch.int32)[: n * 96].view(n, 96)[:, 91], want[2])
    # room for the first chunk of a ray, and for half of the others: the rest of the notes is lost, and the gradient marches
    marched = run(END_TO_END, lambda: C.volume_render_backward(plain, rs, opt, go, workspace=False))
    picture = run(END_TO_END, lambda: C.volume_render(plain, rs, opt))
    for records in (15, 15 * (chunks // 2 + 1)):

        def short():
            out, notes = C.volume_render_noted(plain, rs, opt, records_per_ray=records)
            count = notes.view(torch.int32)[: n * 96].view(n, 96)[:, 91].clone()
            return out, count, C.volume_render_backward_noted(plain, rs, opt, go, notes)
        out, count, grad = run(cut(per_wave, most), short)
        assert torch.equal(out, picture)
        lost = count == -1
        assert torch.equal(count[~lost], want[2][~lost])
        if records == 15:
            assert torch.equal(lost, want[2] > 15)
            assert bool(lost.any()) == (kind != "leaf")
        err, ok = grad_close(grad.cpu().numpy(), marched.cpu().numpy(), slack=slack, what="lost notes")
        assert ok, (records, err)


@pytest.mark.parametrize("ndc", [False, True])
def test_pictures_in_pieces_and_the_sizes_that_take_them(gpu, ndc):
    """The sizes around which the launcher changes over, one picture and several; a captured pass, replayed."""
    tree = synth.shell_tree(depth=6, data_format="SH4", n_spheres=6, seed=4)
    if ndc:
        tree.invradius.fill_(0.5)
        tree.offset.fill_(0.5)
    dev = on_gpu(tree, gpu)
    spec = dev._spec()
    poses = torch.stack(synth.orbit_poses(3, seed=2, radius=3.0))
    if ndc:
        poses = torch.cat([torch.eye(3).expand(3, 3, 3), torch.tensor([[0.1, 0.0, 0.2]]).expand(3, 3)[:, :, None]], dim=2)
    for w, h, k in ((1, 1, 1), (64, 64, 1), (65, 63, 1), (91, 90, 1), (64, 64, 3), (128, 96, 1), (128, 97, 1)):
        opt = options(tree, step_size=1e-3, ndc=svox.NDCConfig(w, h, 0.8 * w) if ndc else None)
        cam = cam_spec(poses[:k].contiguous() if k > 1 else poses[0].contiguous(), w, h, 1.4 * w if not ndc else 0.8 * w, device=gpu)
        f = C.volume_render_images if k > 1 else C.volume_render_image
        want = run(END_TO_END, lambda: f(spec, cam, opt))
        assert torch.equal(f(spec, cam, opt), want)
        out, notes = C.volume_render_images_noted(spec, cam, opt)
        assert torch.equal(out.reshape(want.shape), want)
    rs = rays_spec(synth.sphere_rays(2000, seed=1), gpu)
    opt = options(tree, step_size=1e-3)
    want = run(END_TO_END, lambda: C.volume_render(spec, rs, opt))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        C.volume_render(spec, rs, opt)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = C.volume_render(spec, rs, opt)
    for _ in range(4):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(C.volume_render(spec, rs, opt), want)


@pytest.mark.parametrize("per_wave,most", [(16, 2), (8, 3), (5, 6), (2, 5), (1, 6)])
@pytest.mark.parametrize("kind,fmt,kw", [("dense", "SH9", {}), ("full", "SH4", {"density_softplus": True}), ("full", "SH1", {}), ("deep", "SH4", {}),
                                         ("leaf", "RGBA", {}), ("dense", "SH4", {"fast": True, "min_comp": 1, "max_comp": 2})])
def test_double_precision_rays_in_pieces(gpu, kind, fmt, kw, per_wave, most):
    """Room for the lists of some rays from end to end, of none (every leaf of 64^3 has density), and of trees deeper than the integer
    coordinates: the kernels with one ray per lane are the reference, bit for bit where the sums have one order."""
    n = 333
    gen = torch.Generator().manual_seed(9)
    if kind == "full":
        tree = svox.N3Tree(N=2, data_format=fmt, init_refine=5)
        tree.data.data.normal_(generator=gen)
        tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 0.2 + 0.01
    elif kind == "deep":
        tree = synth.deep_tree(27, data_format=fmt, seed=5)[0]
    else:
        tree = scene(kind, fmt, gen)
    tree = tree.double()
    rays = synth.sphere_rays(n, seed=8, dtype=torch.float64)
    rays.dirs[::7] *= -1.0
    opt = options(tree, step_size=1e-3, **kw)
    spec, rs = on_gpu(tree, gpu)._spec(), rays_spec(rays, gpu)
    go = torch.randn(n, 3, generator=gen, dtype=torch.float64).to(gpu)

    def passes():
        return C.volume_render(spec, rs, opt), C.volume_render_backward(spec, rs, opt, go)

    want, got = run(1, passes), run(32 | (per_wave + 100 * most) << 8, passes)
    assert torch.equal(got[0], want[0])
    # (sums of at most 333 terms in another order: 333 * 2^-53 of their absolute sum each)
    assert (got[1] - want[1]).abs().max() <= 1e-11 * want[1].abs().max()


@pytest.mark.parametrize("n", [40960, 40961])
def test_double_precision_batches_on_either_side_of_the_rule(gpu, n):
    tree = synth.shell_tree(depth=5, n_spheres=5, data_format="SH4", seed=7).double()
    rs = rays_spec(synth.sphere_rays(n, seed=3, dtype=torch.float64), gpu)
    spec, opt = on_gpu(tree, gpu)._spec(), options(tree, step_size=1e-3)
    assert torch.equal(C.volume_render(spec, rs, opt), run(1, lambda: C.volume_render(spec, rs, opt)))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_many_pieces_are_not_walked_in_vain(gpu, dtype):
    """64 pieces to a ray and 32 of each of two rays take times of one kind: a lane that walks to the next piece's samples links up
    with them.  (1 000 rays of a 256^3 SH9 shell in double precision: 95 and 80 us; 323 us where such lanes passed over the pieces ahead of them.)"""
    tree = synth.shell_tree(depth=8, data_format="SH9", n_spheres=24, seed=0)
    rs = rays_spec(synth.sphere_rays(1000, seed=5, dtype=dtype), gpu)
    opt = options(tree, step_size=5e-4)
    spec = on_gpu(tree.to(dtype), gpu)._spec()
    flags = {64: cut(1, 6), 32: cut(2, 5)} if dtype == torch.float32 else {64: 32 | 601 << 8, 32: 32 | 502 << 8}
    times = {64: [], 32: []}
    for _ in range(7):
        for pieces, f in flags.items():
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

            def passes():
                begin.record()
                for _ in range(5):
                    C.volume_render(spec, rs, opt)
                end.record()
            run(f, passes)
            end.synchronize()
            times[pieces].append(begin.elapsed_time(end))
    many, fewer = (sorted(times[k])[3] for k in (64, 32))
    print(f"[pieces] {dtype}: 64 to a ray {many * 200:.0f} us, 32 {fewer * 200:.0f} us", flush=True)
    assert many <= 2 * fewer


@pytest.mark.parametrize("levels,n", [(2, 2560), (3, 14336), (3, 14337), (3, 20480), (3, 20481), (4, 8193), (4, 14337), (4, 20481), (4, 70001), (5, 20480), (5, 20481),
                                      (5, 24577), (5, 32769), (5, 40961), (6, 1281), (6, 16385), (6, 20481), (6, 32769), (1, 2560), (1, 2561)])
def test_double_precision_rules(gpu, levels, n):
    """On either side of the lines between the splits, and between pieces and lanes that walk a ray together."""
    gen = torch.Generator(device=gpu).manual_seed(levels)
    tree = svox.N3Tree(N=2, data_format="SH1", init_refine=levels, device=gpu, dtype=torch.float64)
    tree.data.data.normal_(generator=gen)
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 0.2 + 0.01
    rs, opt, spec = rays_spec(synth.sphere_rays(n, seed=3, dtype=torch.float64), gpu), options(tree, step_size=1e-3), tree._spec()
    go = torch.randn(n, 3, generator=gen, device=gpu, dtype=torch.float64)
    want, ref = run(1, lambda: (C.volume_render(spec, rs, opt), C.volume_render_backward(spec, rs, opt, go)))
    assert torch.equal(C.volume_render(spec, rs, opt), want)
    # (up to n terms of a leaf in another order: n * 2^-53 of the sum of their sizes at most, which cancels to a hundredth of it)
    got = C.volume_render_backward(spec, rs, opt, go)
    assert (got - ref).abs().max() <= n * 1.2e-14 * ref.abs().max()


@pytest.mark.parametrize("gradient,n", [(False, 40960), (True, 131072)])
def test_full_trees_in_double_precision_take_the_faster_kernel(gpu, gradient, n):
    """Every leaf of a 128^3 grid has density: lists of pieces run over, and lanes that walk a ray together are faster.  (Forward pass of
    40 960 rays 670 us, in pieces 1 056; gradient of 131 072 rays 6 338, in pieces 7 670 us.)"""
    tree = svox.N3Tree(N=2, data_format="SH4", init_refine=6, device=gpu, dtype=torch.float64)
    tree.data.data.normal_(generator=torch.Generator(device=gpu).manual_seed(2))
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 0.1 + 0.01
    rs, opt, spec = rays_spec(synth.sphere_rays(n, seed=3, dtype=torch.float64), gpu), options(tree, step_size=1e-3), tree._spec()
    go = torch.randn(n, 3, device=gpu, dtype=torch.float64)
    times = {"rule": [], "pieces": []}
    for _ in range(5):
        for way, flags in (("rule", 0), ("pieces", 32 | 604 << 8)):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

            def passes():
                begin.record()
                for _ in range(2):
                    C.volume_render_backward(spec, rs, opt, go) if gradient else C.volume_render(spec, rs, opt)
                end.record()
            run(flags, passes)
            end.synchronize()
            times[way].append(begin.elapsed_time(end))
    rule, pieces = (sorted(times[k])[2] for k in ("rule", "pieces"))
    print(f"[double] {n} rays, gradient {gradient}: {rule * 500:.0f} us, in pieces {pieces * 500:.0f} us", flush=True)
    assert rule <= 0.92 * pieces


@pytest.mark.parametrize("levels,fmt,n,noted", [(2, "SH1", 4096, False), (6, "SH4", 10000, True), (5, "SH9", 0, True)])
def test_full_trees_are_not_slower_in_pieces(gpu, levels, fmt, n, noted):
    """Trees without empty leaves, whose lists of pieces run over, and tiny ones.  (End to end, rule before the lines were drawn for them and now, us:
    8^3, 4 096 rays 20, 34, 20; 128^3, 10 000 rays with notes 459, 727, 447; 64^3, a picture of 96 x 128 pixels with notes from close up 189, 352, 191.)"""
    tree = svox.N3Tree(N=2, data_format=fmt, init_refine=levels, device=gpu)
    tree.data.data.normal_(generator=torch.Generator(device=gpu).manual_seed(2))
    tree.data.data[..., -1] = tree.data.data[..., -1].abs() * 0.1 + 0.01
    spec, opt = tree._spec(), options(tree, step_size=1e-3)
    if n:
        rs = rays_spec(synth.sphere_rays(n, seed=5), gpu)
        f = (lambda: C.volume_render_noted(spec, rs, opt)) if noted else (lambda: C.volume_render(spec, rs, opt))
    else:
        cam = cam_spec(synth.orbit_poses(1, seed=1, radius=1.2)[0], 96, 128, 1.39 * 128, device=gpu)
        f = lambda: C.volume_render_images_noted(spec, cam, opt)
    times = {"rule": [], "end to end": []}
    for _ in range(7):
        for way, flags in (("rule", 0), ("end to end", 8)):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

            def passes():
                begin.record()
                for _ in range(20):
                    f()
                end.record()
            run(flags, passes)
            end.synchronize()
            times[way].append(begin.elapsed_time(end))
    rule, marched = (sorted(times[k])[3] for k in ("rule", "end to end"))
    print(f"[pieces] {levels} {n}: {rule * 50:.0f} us, from end to end {marched * 50:.0f} us", flush=True)
    assert rule <= 1.2 * marched
