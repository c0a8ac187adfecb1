"""The gradient of point queries collected row by row (partition_kernels.h), against an exact sum on the CPU.

Bar: 1e-5 of the largest element.
"""
import pytest
import torch

import svox_amd as svox
from svox_amd import csrc as C
from svox_amd import synth
from svox_amd.csrc import _abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,levels,dim,n,spread", [
    (2, 5, 28, 700001, 1.0),         # rows of 16 bytes' multiples
    (2, 4, 49, 300007, 1.0),         # ... and not; many points to a row
    (2, 5, 13, 1200000, 0.05),       # most rows empty, the others full: several rounds to a tile
    (2, 0, 49, 300000, 1.0),         # one node
    (2, 3, 76, 400000, 1e-6),        # all points in one leaf
    (3, 3, 49, 500000, 1.0),         # 27 cells to a node, a number of rows that no tile divides
])
def test_gradient_by_rows(gpu, N, levels, dim, n, spread):
    import ctypes
    tree = svox.N3Tree(N=N, data_dim=dim, init_refine=levels, data_format="RGBA").to(gpu)
    gen = torch.Generator().manual_seed(n)
    points = ((torch.rand(n, 3, generator=gen) - 0.5) * spread + 0.51).to(gpu)
    grad = torch.randn(n, dim, generator=gen).to(gpu)
    spec = C._pack_tree(tree._spec(world=False))
    assert _abi.load_library().svox_query_vertical_backward_workspace_bytes(ctypes.byref(spec), n, dim) > 0
    got = C.query_vertical_backward(tree._spec(world=False), points, grad)
    _, ids = C.query_vertical(tree._spec(world=False), points)
    again = C.query_vertical_backward(tree._spec(world=False), points, grad, ids)   # (the leaves known: nothing is looked up)
    want = torch.zeros(tree.data.numel() // dim, dim, dtype=torch.float64)
    want.index_add_(0, ids.cpu(), grad.double().cpu())
    for g in (got, again):
        assert (g.view(-1, dim).cpu().double() - want).abs().max() <= 1e-5 * want.abs().max()


@pytest.mark.parametrize("n,dtype,N", [(65536, torch.float32, 2), (70001, torch.float64, 2), (300001, torch.float32, 3)])
def test_gradient_at_known_leaves(gpu, n, dtype, N):
    """Atomics at leaves the query kept: both launch shapes, both scalar types; ids that are no cell add nothing; and what
    makes the leaves void (the tree or the ids written to before the backward pass)."""
    tree = svox.N3Tree(N=N, data_dim=4, init_refine=3, data_format="RGBA", dtype=dtype).to(gpu)
    gen = torch.Generator().manual_seed(n)
    points = torch.rand(n, 3, generator=gen, dtype=dtype).to(gpu)
    grad = torch.randn(n, 4, generator=gen, dtype=dtype).to(gpu)
    spec = tree._spec()
    _, ids = C.query_vertical(spec, points)

    def sums(ids):
        want = torch.zeros(tree.data.numel() // 4, 4, dtype=torch.float64)
        ok = (ids >= 0) & (ids < want.shape[0])
        return want.index_add_(0, ids[ok].cpu(), grad[ok].double().cpu())
    odd = ids.clone()
    odd[::7], odd[3::7] = -1, tree.child.numel()
    for known in (ids, odd):
        got = C.query_vertical_backward(spec, points, grad, known).view(-1, 4).cpu().double()
        want = sums(known)
        assert (got - want).abs().max() <= 1e-5 * want.abs().max()
    for void in (False, True):
        tree.data.grad = None
        values, node_ids = tree(points, want_node_ids=True)
        if void:
            node_ids.zero_()
        values.backward(grad)
        want = sums(ids)
        assert (tree.data.grad.view(-1, 4).cpu().double() - want).abs().max() <= 1e-5 * want.abs().max()


def _crowd(gen, n, kind):
    if kind == "space":
        return torch.rand(n, 3, generator=gen)
    if kind == "leaf":
        return torch.rand(n, 3, generator=gen) * 1e-6 + 0.51
    return (torch.randn(n, 3, generator=gen) * 0.1 + 0.5).clamp(0, 1)      # "blob"


@pytest.mark.parametrize("tree,dim,n,kind,shifted", [
    (("shell", 6), 49, 262145, "space", False),    # runs of 512 pairs, rows that no 16-byte piece divides
    (("shell", 8), 28, 800001, "space", False),    # ... of 1 562, 16-byte pieces
    (("shell", 8), 28, 800001, "space", True),     # the same from an address that 16 bytes do not divide
    (("shell", 9), 28, 2200001, "space", False),   # more than 2 048 bins, runs of 4 096
    (("dense", 6), 49, 1000003, "blob", False),    # crowded bins beside others with several rounds to a tile
    (("dense", 6), 28, 1000003, "leaf", False),    # one row has all the pairs of every run
    (("dense", 1), 300, 40000, "blob", False),     # two tiles for everything
])
def test_gradient_by_rows_where_points_crowd(gpu, tree, dim, n, kind, shifted):
    """Values where many points share few rows: crowded bins, their runs and the long rows of tiles, against a sum in double
    precision; and the time, which must not be far from that of atomics (the workspace withheld) wherever the points fall."""
    import ctypes
    gen = torch.Generator().manual_seed(n)
    if tree[0] == "shell":
        tree = synth.shell_tree(depth=tree[1], n_spheres=24, data_format="RGBA", seed=0, device=gpu)
    else:
        tree = svox.N3Tree(data_format="RGBA", init_refine=tree[1] - 1, device=gpu)
    points = _crowd(gen, n, kind).to(gpu)
    grad = torch.randn(n * dim + 1, generator=gen).to(gpu)[int(shifted):][:n * dim].view(n, dim)
    spec = tree._spec(world=False)
    packed = C._pack_tree(spec)
    lib = _abi.load_library()
    need = lib.svox_query_vertical_backward_workspace_bytes(ctypes.byref(packed), n, dim)
    assert need > 0
    _, ids = C.query_vertical(spec, points)
    want = torch.zeros(tree.child.numel(), dim, dtype=torch.float64, device=gpu).index_add_(0, ids, grad.double())
    # (a sum of m terms of about 1 in single precision, in runs, is off by less than sqrt(m) 2^-24 times the largest partial sum)
    for known in (None, ids):
        got = C.query_vertical_backward(spec, points, grad, known).view(-1, dim)
        assert (got.double() - want).abs().max() <= 1e-5 * want.abs().max()
    out = torch.empty(tree.child.numel(), dim, device=gpu)
    space = torch.empty(need, dtype=torch.uint8, device=gpu)
    stream = torch.cuda.current_stream(gpu).cuda_stream
    times = {}
    for way, at, size in [("rows", space.data_ptr(), need), ("atomics", None, 0)] * 8:
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        assert lib.svox_query_vertical_backward_ids(ctypes.byref(packed), points.data_ptr(), ids.data_ptr(), n, grad.data_ptr(), dim,
                                                    out.data_ptr(), 0, at, size, stream) == 0
        end.record()
        end.synchronize()
        times.setdefault(way, []).append(begin.elapsed_time(end) * 1e3)
    rows, atomics = (sorted(times[w])[4] for w in ("rows", "atomics"))
    print(f"[rows] {kind} {n}: by rows {rows:.0f} us, with atomics {atomics:.0f} us", flush=True)
    assert rows <= 1.5 * atomics + 30.0
