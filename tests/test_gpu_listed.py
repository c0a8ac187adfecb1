"""Noting passes that list the rays of a batch, or the pixels of pictures, which meet the tree: two wavefronts per tile, one, or all as they are, whichever the
number of them asks for on the device.

Bar: pictures, noted colours and the number of notes of every ray equal to those of the pass that takes the batch as it is, bit for bit;
gradients the same terms in another order.
"""
import pytest
import torch

import svox_amd as svox
from svox_amd import csrc as C
from svox_amd import synth
from util import cam_spec, grad_close, on_gpu, options, rays_spec

pytestmark = pytest.mark.gpu


def listed(two, one):
    """flags: up to `two` * 64 listed rays on two wavefronts per tile, up to `one` * 64 on one"""
    return 64 | two << 8 | one << 16


def run(flags, f):
    C.set_debug_flags(flags)
    try:
        return f()
    finally:
        C.set_debug_flags(0)


# how many rays meet the tree, of 2 500: none, one, a tile and one more, all
@pytest.mark.parametrize("hits", [0, 1, 64, 65, 1025, 2500])
@pytest.mark.parametrize("two,one,more", [(255, 256, 0), (16, 32, 0), (1, 16, 2), (0, 40, 0), (1, 1, 2)])
def test_listed_rays(gpu, oracle_mod, monkeypatch, hits, two, one, more):
    n = 2500
    tree = synth.shell_tree(depth=6, data_format="SH9", n_spheres=6, seed=4)
    gen = torch.Generator().manual_seed(hits)
    rays = synth.sphere_rays(n, seed=8)
    away = torch.randperm(n, generator=gen)[hits:]
    rays.dirs[away] = rays.origins[away] - 0.5          # (outwards)
    opt = options(tree, step_size=1e-3)
    dev, rs = on_gpu(tree, gpu), rays_spec(rays, gpu)
    spec = dev._spec()
    go, target = (torch.randn(n, 3, generator=gen) * 1e-2).to(gpu), torch.rand(n, 3, generator=gen).to(gpu)
    slack = oracle_mod.volume_render_backward(oracle_mod.Tree.from_n3tree(tree), rays.origins, rays.dirs, rays.viewdirs, opt, go.cpu(),
                                              want_slack=True)[1]

    def passes():
        out, notes = C.volume_render_noted(spec, rs, opt, records_per_ray=64)
        count = notes.view(torch.int32)[: n * 96].view(n, 96)[:, 91].clone()
        return (out, count, C.se_grad(spec, rs, target, opt)[0], C.volume_render_backward_noted(spec, rs, opt, go, notes),
                C.volume_render_backward(spec, rs, opt, go))

    want, got = run(4, passes), run(listed(two, one) | more, passes)
    for what, a, b in zip(("picture", "notes", "colours"), got, want):
        assert torch.equal(a, b), what
    for what, a, b in zip(("from notes", "alone"), got[3:], want[3:]):
        err, ok = grad_close(a.cpu().numpy(), b.cpu().numpy(), slack=slack, what=what)
        assert ok, (what, err)
    # no room for the list beside the notes, and for those of a ray beyond the first 15: the batch as it is
    monkeypatch.setattr(C, "SMALL_BATCH_ROOM", 1)

    def short():
        out, notes = C.volume_render_noted(spec, rs, opt, records_per_ray=15)
        assert notes.numel() * 8 // 384 - n < 16 * (n * 4 // 384)
        count = notes.view(torch.int32)[: n * 96].view(n, 96)[:, 91].clone()
        return out, count, C.volume_render_backward_noted(spec, rs, opt, go, notes)

    out, count, grad = run(listed(two, one) | more, short)
    assert torch.equal(out, want[0])
    assert torch.equal(count, torch.where(want[1] > 15, -1, want[1]))
    assert bool((count == -1).any()) == (hits >= 64)
    err, ok = grad_close(grad.cpu().numpy(), want[3].cpu().numpy(), slack=slack, what="no room")
    assert ok, err


def test_a_captured_pass_lists_anew_in_every_replay(gpu):
    n = 200001
    tree = synth.shell_tree(depth=7, data_format="SH1", n_spheres=6, seed=4)
    dev, rs = on_gpu(tree, gpu), rays_spec(synth.sphere_rays(n, seed=8), gpu)
    spec, opt = dev._spec(), options(tree, step_size=1e-3)
    turned = rs.dirs.clone()
    turned[::3] *= -1.0
    kept = rs.dirs.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        C.volume_render_noted(spec, rs, opt)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, notes = C.volume_render_noted(spec, rs, opt)
    for dirs in (kept, turned, turned, kept):
        rs.dirs.copy_(dirs)
        want = run(4, lambda: C.volume_render_noted(spec, rs, opt)[0])
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(C.volume_render_noted(spec, rs, opt)[0], want)


def test_batches_that_all_hit_are_hardly_slower(gpu):
    """Where most rays of a sample hit, none are listed.  (Noting march of 500 000 rays of a 256^3 shell that all hit: as it is 1096 us, with
    the rule 1105; 1128 where all of them were listed first.)"""
    n = 500000
    tree = synth.shell_tree(depth=8, data_format="SH9", n_spheres=24, seed=0, device=gpu)
    rs, opt, spec = rays_spec(synth.sphere_rays(n, seed=5), gpu), options(tree, step_size=5e-4), tree._spec()
    times = {0: [], 4: []}
    for _ in range(7):
        for flags in times:
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

            def passes():
                begin.record()
                for _ in range(20):
                    C.volume_render_noted(spec, rs, opt)
                end.record()
            run(flags, passes)
            end.synchronize()
            times[flags].append(begin.elapsed_time(end))
    rule, plain = (sorted(times[k])[3] for k in (0, 4))
    print(f"[listed] all hit: {rule * 50:.0f} us, as it is {plain * 50:.0f} us", flush=True)
    assert rule <= 1.018 * plain


def test_pictures_leave_no_room_for_a_list(gpu):
    """All chunks of a picture's workspace are for notes; of a batch of as many rays, a number per ray is taken off."""
    w, h = 512, 300
    n = w * h
    tree = synth.shell_tree(depth=5, data_format="SH1", n_spheres=6, seed=4)
    spec, opt = on_gpu(tree, gpu)._spec(), options(tree, step_size=1e-3)
    cam = cam_spec(synth.orbit_poses(1, seed=2, radius=3.0)[0], w, h, 1.4 * w, device=gpu)
    go = torch.ones(n, 3, device=gpu) * 1e-2
    report = torch.zeros(1, dtype=torch.int64, pin_memory=True)
    chunks = lambda notes: (notes.numel() * 8 - 256 - 16 * ((n + 127) // 128)) // 384

    notes = C.volume_render_images_noted(spec, cam, opt, records_per_ray=30)[1]
    C.volume_render_images_backward_noted(spec, cam, opt, go.view(h, w, 3), notes, report.data_ptr())
    torch.cuda.synchronize()
    assert int(report[0]) & 0xffffffff == (chunks(notes) - n + 63) // 64
    rs = rays_spec(synth.sphere_rays(n, seed=8), gpu)
    notes = C.volume_render_noted(spec, rs, opt, records_per_ray=30)[1]
    C.volume_render_backward_noted(spec, rs, opt, go, notes, report.data_ptr())
    torch.cuda.synchronize()
    assert int(report[0]) & 0xffffffff == (chunks(notes) - -(-n * 4 // 384) - n + 63) // 64 == C.notes_pool_use(notes, n)[1]


# pictures: of which no pixel meets the tree, some, all; pieces of 16 pixels with a rest and without; one and several; listed, or more than are
@pytest.mark.parametrize("w,h,n_images", [(16, 1, 1), (33, 31, 1), (48, 40, 2), (100, 67, 3), (128, 96, 1)])
@pytest.mark.parametrize("view", ["none", "some", "all"])
@pytest.mark.parametrize("tiles", [255, 1])
def test_listed_pixels(gpu, oracle_mod, w, h, n_images, view, tiles):
    n = w * h * n_images
    tree = synth.shell_tree(depth=6, data_format="SH9", n_spheres=6, seed=4)
    gen = torch.Generator().manual_seed(n)
    poses = torch.stack([p[:3] for p in synth.orbit_poses(n_images, seed=2, radius=3.0)])
    poses[:, :, 3] += 100.0 if view == "none" else 0.0
    fx = 1.1 * w if view == "some" else 12.0 * w
    opt = options(tree, step_size=1e-3)
    dev = on_gpu(tree, gpu)
    spec = dev._spec()
    cam, one = cam_spec(poses, w, h, fx, device=gpu), cam_spec(poses[0], w, h, fx, device=gpu)
    go, target = (torch.randn(n_images, h, w, 3, generator=gen) * 1e-2).to(gpu), torch.rand(h, w, 3, generator=gen).to(gpu)
    slack = sum(oracle_mod.volume_render_image_backward(oracle_mod.Tree.from_n3tree(tree), p, fx, fx, w, h, opt, g, want_slack=True)[1]
                for p, g in zip(poses, go.cpu()))

    def passes():
        out, notes = C.volume_render_images_noted(spec, cam, opt, records_per_ray=64)
        count = notes.view(torch.int32)[: n * 96].view(n, 96)[:, 91].clone()
        hit = notes.view(torch.float32)[: n * 96].view(n, 96)[:, 93] != 1.0
        assert {"none": bool(~hit.any()), "some": bool(hit.any()) and not bool(hit.all()) or n == 16, "all": bool(hit.all())}[view]
        number = C.notes_pool_use(notes, n)[0]
        said = int(notes.view(torch.int64)[number.storage_offset() + 2])
        return (out, count, C.se_grad_persp(spec, one, opt, target)[0], said, int(hit.sum()), C.volume_render_images_backward_noted(spec, cam, opt, go, notes),
                C.volume_render_images_backward(spec, cam, opt, go))

    want, got = run(8, passes), run(64 | tiles << 8, passes)
    for what, a, b in zip(("pictures", "notes", "colours"), got, want):
        assert torch.equal(a, b), what
    assert want[3] == 0 and got[3] in (got[4], n)
    for what, a, b in zip(("from notes", "alone"), got[5:], want[5:]):
        err, ok = grad_close(a.cpu().numpy(), b.cpu().numpy(), slack=slack, what=what)
        assert ok, (what, err)


@pytest.mark.parametrize("w", [128, 200, 361, 363])
@pytest.mark.parametrize("fx", [1.39, 4.0])
@pytest.mark.parametrize("records", [30, 300])
def test_the_pool_of_a_picture_of_any_size(gpu, monkeypatch, w, fx, records):
    """svox_notes_pool_info knows the number of rays and no more: of pictures with fewer than 131 072 pixels, which are listed where a batch of as
    many rays is not, and of larger ones (363 x 363), it says what the pass and its replay go by, and a count below that says that no note was lost."""
    monkeypatch.setattr(C, "SMALL_BATCH_ROOM", 1)
    n = w * w
    tree = synth.shell_tree(depth=7, data_format="SH9", n_spheres=24, seed=0, device=gpu)
    spec, opt = tree._spec(), options(tree, step_size=5e-4)
    cam = cam_spec(synth.orbit_poses(1, seed=2, radius=4.0)[0], w, w, fx * w, device=gpu)
    report = torch.zeros(1, dtype=torch.int64, pin_memory=True)
    got = []
    for flags in (0, 8):
        out, notes = run(flags, lambda: C.volume_render_images_noted(spec, cam, opt, records_per_ray=records))
        counter, pool = C.notes_pool_use(notes, n)
        asked, listed = (int(v) for v in notes.view(torch.int64)[counter.storage_offset():][[0, 2]])
        count = notes.view(torch.int32)[: n * 96].view(n, 96)[:, 91].clone()
        grad = run(flags, lambda: C.volume_render_images_backward_noted(spec, cam, opt, torch.ones_like(out), notes, report.data_ptr()))
        torch.cuda.synchronize()
        if flags == 0:
            assert int(report[0]) == asked << 32 | pool and listed > 0
            assert asked <= pool or bool((count < 0).any())      # (the last stock may be a part of one)
        assert asked >= pool or bool((count >= 0).all())
        got.append((out, count, grad, asked))
    assert torch.equal(got[0][0], got[1][0])
    if records == 300:
        assert torch.equal(got[0][1], got[1][1])
    err, ok = grad_close(got[0][2].cpu().numpy(), got[1][2].cpu().numpy())
    assert ok, err


@pytest.mark.parametrize("N,levels", [(3, 3), (4, 2)])
def test_pictures_of_other_branching_factors_are_not_listed(gpu, N, levels):
    tree = svox.N3Tree(N=N, data_format="SH1", init_refine=levels, device=gpu)
    tree.data.data[..., -1] = 1.0
    w = 150
    spec, opt = tree._spec(), options(tree, step_size=1e-3)
    cam = cam_spec(synth.orbit_poses(1, seed=2, radius=4.0)[0], w, w, 1.39 * w, device=gpu)
    for flags, listed in ((0, False), (64 | 255 << 8, True)):
        notes = run(flags, lambda: C.volume_render_images_noted(spec, cam, opt)[1])
        counter = C.notes_pool_use(notes, w * w)[0]
        assert bool(notes.view(torch.int64)[counter.storage_offset() + 2] > 0) == listed


def test_the_rule_lists_pictures_of_shells(gpu):
    """Where the rule says so the pixels are listed, all that meet the cube, and the last of the chunks are not for notes.  (400x400 picture of a 256^3
    SH9 shell, noting march 307 us as it is, 252 listed.)"""
    w = 400
    tree = synth.shell_tree(depth=8, data_format="SH9", n_spheres=24, seed=0, device=gpu)
    spec, opt = tree._spec(), options(tree, step_size=5e-4)
    cam = cam_spec(synth.orbit_poses(1, seed=2, radius=4.0)[0], w, w, 1.39 * w, device=gpu)
    out, notes = C.volume_render_images_noted(spec, cam, opt, records_per_ray=30)
    counter, pool = C.notes_pool_use(notes, w * w)
    listed = int(notes.view(torch.int64)[counter.storage_offset() + 2])
    head = notes.view(torch.float32)[: w * w * 96].view(w * w, 96)
    assert int((head[:, 93] != 1.0).sum()) <= listed < w * w
    report = torch.zeros(1, dtype=torch.int64, pin_memory=True)
    C.volume_render_images_backward_noted(spec, cam, opt, torch.ones_like(out), notes, report.data_ptr())
    torch.cuda.synchronize()
    assert int(report[0]) & 0xffffffff == pool
    assert torch.equal(out, run(8, lambda: C.volume_render_images_noted(spec, cam, opt, records_per_ray=30)[0]))
