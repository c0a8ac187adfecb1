"""Walk tables: the child table made over for the march (a node that has leaves only is known by the entry that leads to it)."""
import ctypes

import numpy as np
import pytest
import torch

import svox_amd as svox
from svox_amd import csrc as C
from svox_amd import synth
from svox_amd.csrc import _abi
from util import grad_close, on_gpu, options, rays_spec

ALWAYS = 128      # debug flag: every call that could makes one


def test_which_calls_make_a_walk_table():
    lib = _abi.load_library()
    spec, opt = _abi.TreeSpecC(), _abi.RenderOptionsC()
    spec.data = spec.child = spec.parent_depth = 16
    spec.N, spec.data_dim, spec.dtype = 2, 13, 0
    opt.format, opt.basis_dim, opt.max_comp, opt.ndc_width = 1, 4, 3, -1

    def first(nodes, image, positive, low=1, high=1 << 30):
        spec.capacity = nodes
        ask = lambda n: lib.svox_walk_table_bytes(ctypes.byref(spec), ctypes.byref(opt), n, image, positive)
        assert all(ask(n) in (0, nodes * 32) for n in (1, 20000, 1 << 20, 1 << 24))
        while low < high:
            middle = (low + high) // 2
            low, high = (low, middle) if ask(middle) > 0 else (middle + 1, high)
        return low

    grid64, grid128, shell = 37449, 299593, 192314
    assert first(grid64, 0, 0) == first(grid64, 0, 1) == first(grid128, 0, 0) == 12289
    assert first(shell, 0, 1) == 40000 and first(shell, 0, 0) == 65536 and first(shell, 1, 0) == 12289
    assert first(4681, 0, 1) == first(grid64, 1, 0) == 1 << 30 and first(grid128, 1, 0, high=262144) == 12289
    assert first((1 << 22) - 1, 1, 0) == 12289 and first(1 << 22, 1, 0) == 1 << 30      # (a node's number has 22 bits)
    assert first(shell, 1, 1) == 12289 and first(47433, 1, 1) == first(grid128, 1, 1) == 1 << 30
    opt.ndc_width = 100
    assert first(shell, 1, 0, high=65536) == 12289
    opt.ndc_width, opt.density_softplus = -1, 1
    assert first(shell, 1, 0) == first(shell, 0, 0) == first(grid128, 1, 0) == first(grid128, 0, 1) == 1 << 30 and first(grid64, 0, 0) == 12289
    opt.density_softplus = 0
    opt.ndc_width, spec.N = -1, 3
    assert first(shell, 0, 1) == 1 << 30


def test_tables_that_do_not_begin_at_16_bytes_serve_no_walk_table():
    lib = _abi.load_library()
    spec, opt = _abi.TreeSpecC(), _abi.RenderOptionsC()
    spec.data = spec.parent_depth = 16
    spec.capacity, spec.N, spec.data_dim, spec.dtype = 192314, 2, 13, 0
    opt.format, opt.basis_dim, opt.max_comp, opt.ndc_width, opt.sigma_thresh = 1, 4, 3, -1, 0.0
    made = _abi.TreeSpecC()
    for always in (0, ALWAYS):
        C.set_debug_flags(always)
        try:
            # (marks that do not apply to the call, softened ones here, are not what the table is made from)
            for child, marks, softened, pays in ((4096, 0, 0, True), (4100, 0, 0, False), (4104, 0, 0, False), (4100, 8192, 0, True), (4096, 8196, 0, False),
                                                 (4096, 8196, 1, True), (4100, 8192, 1, False)):
                spec.child, spec.child_marks, spec.child_marks_softplus = child, marks, softened
                assert lib.svox_walk_table_bytes(ctypes.byref(spec), ctypes.byref(opt), 1 << 20, 1, 0) == (192314 * 32 if pays else 0), (child, marks)
                if not pays:
                    assert lib.svox_walk_table(ctypes.byref(spec), ctypes.byref(opt), 0, 4096, ctypes.byref(made), None) == -2
        finally:
            C.set_debug_flags(0)


@pytest.mark.gpu
def test_a_child_table_that_does_not_begin_at_16_bytes(gpu):
    tree = synth.shell_tree(depth=8, data_format="SH1", n_spheres=24, seed=0, device=gpu)
    rs, opt, spec = rays_spec(synth.sphere_rays(70001, seed=4), gpu), options(tree, step_size=1e-3), tree._spec()
    want = C.volume_render(spec, rs, opt)
    room = torch.empty(spec.child.numel() + 1, dtype=torch.int32, device=gpu)
    room[1:] = spec.child.flatten()
    spec.child = room[1:].view(spec.child.shape)
    assert spec.child.data_ptr() % 16 == 4 and torch.equal(C.volume_render(spec, rs, opt), want)


@pytest.mark.gpu
def test_a_picture_of_a_small_tree_with_marks_is_marched_on_them(gpu):
    """Allocations of a call: what it returns, and a walk table."""
    tree = synth.shell_tree(depth=7, data_format="SH1", n_spheres=24, seed=0, device=gpu)
    opt, spec = options(tree, step_size=1e-3, fast=True), tree._spec()
    poses = torch.stack(synth.orbit_poses(2, seed=1, radius=4.0)).contiguous().to(gpu)
    marks = C.mark_empty_leaves(spec, opt.sigma_thresh, False)
    for n, marked, made in ((1, False, 2), (1, True, 1), (2, False, 2), (2, True, 2)):
        spec.child_marks, spec.child_marks_thresh = (marks, opt.sigma_thresh) if marked else (None, 0.0)
        cam = C.CameraSpec()
        cam.c2w, cam.fx, cam.fy, cam.width, cam.height = poses[:n], 170.0, 170.0, 128, 128
        before = torch.cuda.memory_stats(gpu)["allocation.all.allocated"]
        C.volume_render_images(spec, cam, opt)
        assert torch.cuda.memory_stats(gpu)["allocation.all.allocated"] - before == made, (n, marked)


@pytest.mark.gpu
def test_calls_without_memory_for_a_walk_table_do_without(gpu):
    """The table takes 6 MB, for which torch asks for 20; the picture fits 2."""
    tree = synth.shell_tree(depth=8, data_format="SH1", n_spheres=24, seed=0, device=gpu)
    rs, opt, spec = rays_spec(synth.sphere_rays(70001, seed=4), gpu), options(tree, step_size=1e-3), tree._spec()
    want = C.volume_render(spec, rs, opt)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(gpu).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(gpu) + (6 << 20)) / total, gpu)
    held = []
    try:
        with pytest.raises(torch.OutOfMemoryError):
            # (what is left of the blocks there are)
            for _ in range((torch.cuda.memory_reserved(gpu) - torch.cuda.memory_allocated(gpu)) // (tree.child.numel() * 4) + 20):
                held.append(torch.empty(tree.child.numel(), dtype=torch.int32, device=gpu))
        got = C.volume_render(spec, rs, opt)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu)
    assert torch.equal(got, want)


@pytest.mark.parametrize("softplus", [0, 1, 2, 3, 4, 6, 7, -1])
def test_any_number_but_0_says_that_marks_are_softened(softplus):
    """... and none that they are a walk table, of which no second one is made."""
    lib = _abi.load_library()
    spec, opt = _abi.TreeSpecC(), _abi.RenderOptionsC()
    spec.data = spec.child = spec.parent_depth = spec.child_marks = 16
    spec.capacity, spec.N, spec.data_dim, spec.dtype = 192314, 2, 13, 0
    opt.format, opt.basis_dim, opt.max_comp, opt.ndc_width = 1, 4, 3, -1
    spec.child_marks_softplus = softplus
    for thresh in (0.0, -0.0, 1e-2, float("inf")):
        spec.child_marks_thresh = thresh
        assert lib.svox_walk_table_bytes(ctypes.byref(spec), ctypes.byref(opt), 1 << 20, 1, 0) == 192314 * 32, thresh


@pytest.mark.gpu
@pytest.mark.parametrize("softplus", [1, 2, 3, 6, -1])
@pytest.mark.parametrize("thresh", [0.0, 0.6])
def test_marks_with_softplus_whatever_number_says_so(gpu, softplus, thresh):
    """Marks, and walk tables made from them; a call to which they do not apply leaves them aside."""
    tree = grown(2)
    # (softened, -200 is 0, and 0.7 less than 0.6)
    some = torch.rand(tree.child.shape, generator=torch.Generator().manual_seed(7))
    tree.data.data[..., -1][some < 0.2] = -200.0
    tree.data.data[..., -1][some > 0.8] = 0.7
    rs, spec = rays_spec(synth.sphere_rays(1500, seed=4), gpu), on_gpu(tree, gpu)._spec()
    rays = C._pack_rays(rs, torch.float32)
    for soft in (True, False):
        opt = options(tree, step_size=1e-3, sigma_thresh=thresh, density_softplus=soft)
        want = C.volume_render(spec, rs, opt)
        grad = C.volume_render_backward(spec, rs, opt, want, workspace=False)
        packed, marks = C._pack_tree(spec), C.mark_empty_leaves(spec, thresh, True)
        assert int((marks < 0).sum()) > marks.numel() // 10
        packed.child_marks, packed.child_marks_thresh, packed.child_marks_softplus = marks.data_ptr(), thresh, softplus
        table, made = torch.empty_like(marks), _abi.TreeSpecC()
        stream = torch.cuda.current_stream().cuda_stream
        for positive in (0, 1):
            C._call("svox_walk_table", ctypes.byref(packed), ctypes.byref(opt._pack()), positive, table.data_ptr(), ctypes.byref(made), stream)
            applies = soft and (thresh == 0.0 or not positive)
            assert made.child_marks_softplus == (3 if applies else 6)
            for kernel in (4, 8):
                C.set_debug_flags(kernel)
                try:
                    for given in (packed, made):
                        out, again = torch.empty_like(want), torch.empty_like(grad)
                        C._call("svox_volume_render", ctypes.byref(given), ctypes.byref(rays), ctypes.byref(opt._pack()), out.data_ptr(), stream)
                        C._call("svox_volume_render_backward", ctypes.byref(given), ctypes.byref(rays), ctypes.byref(opt._pack()),
                                want.data_ptr(), again.data_ptr(), 0, stream)
                        assert torch.equal(out, want), (soft, kernel)
                        # (the same terms in another order, as above)
                        assert (again - grad).abs().max() <= 2e-4 * grad.abs().max(), (soft, kernel)
                finally:
                    C.set_debug_flags(0)


def grown(seed, steps=6):
    """A tree refined a few leaves at a time, so that its nodes lie in no order, with empty leaves and full ones."""
    g = torch.Generator().manual_seed(seed)
    tree = svox.N3Tree(N=2, data_format="SH1", init_refine=1)
    for _ in range(steps):
        leaves = tree._all_leaves()
        pick = leaves[torch.randperm(len(leaves), generator=g)[:24]]
        tree.refine(sel=tuple(pick.T))
    tree.data.data.copy_(torch.randn(tree.data.shape, generator=g))
    tree.data.data[..., -1] = 20 * torch.rand(tree.child.shape, generator=g) * (torch.rand(tree.child.shape, generator=g) < 0.4)
    return tree


def trees():
    yield "one node", svox.N3Tree(N=2, data_format="SH1", init_refine=0)
    yield "grown", grown(1)
    yield "shell", synth.shell_tree(depth=6, n_spheres=4, data_format="SH4", seed=1)
    for levels in (12, 27):
        yield f"deep {levels}", synth.deep_tree(levels, data_format="SH1", seed=levels)[0]


@pytest.mark.gpu
@pytest.mark.parametrize("marks", [False, True])
def test_what_a_walk_table_holds(gpu, marks):
    for name, tree in trees():
        dev = on_gpu(tree, gpu)
        opt = options(dev, step_size=1e-3, sigma_thresh=0.0)
        spec = dev._spec()
        if marks:
            spec.child_marks = C.mark_empty_leaves(spec, 0.0, False)
        table = torch.full((dev.child.numel(),), 7, dtype=torch.int32, device=gpu)
        made = _abi.TreeSpecC()
        packed = C._pack_tree(spec)
        C._call("svox_walk_table", ctypes.byref(packed), ctypes.byref(opt._pack()), 0, table.data_ptr(), ctypes.byref(made),
                torch.cuda.current_stream().cuda_stream)
        got = table.cpu().numpy().astype(np.int64) & 0xffffffff
        rows = (spec.child_marks if marks else dev.child).cpu().numpy().reshape(-1, 8).astype(np.int64)
        bits = ((rows < 0) << np.arange(8)).sum(1)
        last = (rows <= 0).all(1)
        for node, row in enumerate(rows):
            for cell, c in enumerate(row):
                want = 0 if c == 0 else 0x80000000 | 255 << 22
                if c > 0:
                    want = c | (1 << 30 | int(bits[node + c]) << 22 if last[node + c] else 0)
                if last[node] and node > 0:
                    want = 7      # (read by nobody)
                assert got[node * 8 + cell] == want, (name, node, cell)
        assert made.child_marks == table.data_ptr() and made.child_marks_softplus == (2 if marks else 6)


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", [4, 8, 2, 32 | 24 << 8, 64 | 1 << 8 | 2 << 16])
def test_walks_on_a_walk_table_are_those_on_the_child_table(gpu, oracle_mod, kernel):
    """One wavefront per tile, two, wavefronts that take new rays, rays in pieces (which are given the table and leave it aside: they walk on the child
    table alone), listed rays; with marks and without."""
    for name, tree in trees():
        if name == "one node":
            tree.data.data.copy_(torch.rand(tree.data.shape, generator=torch.Generator().manual_seed(3)) * 2)
        ot = oracle_mod.Tree.from_n3tree(tree)
        dev = on_gpu(tree, gpu)
        rays = synth.sphere_rays(1500, seed=4)
        rs = rays_spec(rays, gpu)
        go = torch.randn(1500, 3, generator=torch.Generator().manual_seed(5))
        for thresh, softplus, marked in ((1e-2, False, False), (1e-2, False, True), (0.0, False, True), (0.0, True, False)):
            opt = options(tree, step_size=1e-3, sigma_thresh=thresh, density_softplus=softplus)
            spec = dev._spec()
            if marked:
                spec.child_marks, spec.child_marks_thresh = C.mark_empty_leaves(spec, thresh, False), thresh
            ref = oracle_mod.volume_render(ot, rays.origins, rays.dirs, rays.viewdirs, opt)
            C.set_debug_flags(kernel | ALWAYS)
            try:
                out = C.volume_render(spec, rs, opt).cpu().numpy()
                noted, notes = C.volume_render_noted(spec, rs, opt)
                grad = C.volume_render_backward_noted(spec, rs, opt, go.to(gpu), notes).cpu().numpy()
                marched = C.volume_render_backward(spec, rs, opt, go.to(gpu), workspace=False).cpu().numpy()
                alone = C.volume_render_backward(spec, rs, opt, go.to(gpu)).cpu().numpy()
                squared = C.se_grad(spec, rs, ref_colour(gpu), opt)
            finally:
                C.set_debug_flags(0)
            if softplus:      # (logf is the platform's)
                assert np.abs(out - ref).max() <= 1e-5
            else:
                assert np.array_equal(out, ref), (name, thresh, marked)
            assert np.array_equal(noted.cpu().numpy(), out)
            plain = dev._spec()
            want = C.volume_render_backward(plain, rs, opt, go.to(gpu), workspace=False).cpu().numpy()
            # (the same terms in other orders)
            scale = np.abs(want).max() + 1e-30
            for got in (grad, marched, alone):
                assert np.abs(got - want).max() <= 2e-4 * scale, (name, thresh, softplus, marked)
            again = C.se_grad(plain, rs, ref_colour(gpu), opt)
            assert torch.equal(squared[0], again[0])
            for a, b in zip(squared[1:], again[1:]):
                assert (a - b).abs().max() <= 2e-4 * b.abs().max() + 1e-30


def ref_colour(gpu):
    return torch.rand(1500, 3, generator=torch.Generator().manual_seed(6)).to(gpu)


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", [4, 8, 32 | 24 << 8])
@pytest.mark.parametrize("thresh,marked", [(1e-2, False), (1e-2, True), (0.0, True)])
@pytest.mark.parametrize("fx", [90.0, 700.0, 4000.0])
def test_pictures_on_a_walk_table(gpu, oracle_mod, kernel, thresh, marked, fx):
    """From afar, and from where some tiles' rays, or all, run so close together that they walk on the child table."""
    tree = synth.shell_tree(depth=7, n_spheres=6, data_format="SH9", seed=2)
    dev = on_gpu(tree, gpu)
    poses = torch.stack(synth.orbit_poses(2, seed=1, radius=2.5)).contiguous().to(gpu)
    opt = options(tree, step_size=1e-3, sigma_thresh=thresh)
    spec = dev._spec()
    cam = C.CameraSpec()
    cam.c2w, cam.fx, cam.fy, cam.width, cam.height = poses, fx, fx, 61, 45
    want = C.volume_render_images(spec, cam, opt)
    if marked:
        spec.child_marks, spec.child_marks_thresh = C.mark_empty_leaves(spec, thresh, False), thresh
    C.set_debug_flags(kernel | ALWAYS)
    try:
        got = C.volume_render_images(spec, cam, opt)
        noted, notes = C.volume_render_images_noted(spec, cam, opt)
    finally:
        C.set_debug_flags(0)
    assert torch.equal(got, want) and torch.equal(noted, want)
