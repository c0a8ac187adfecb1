"""The operators and Python's threads."""
import subprocess
import threading
import time

import pytest
import torch

import svox_amd as svox
from svox_amd import csrc as C
from svox_amd import synth
from svox_amd.csrc import _abi
from util import options, rays_spec

pytestmark = pytest.mark.gpu

WAITING = ["svox_query_vertical_ws", "svox_query_vertical_backward_ids", "svox_volume_render", "svox_volume_render_backward_ws",
           "svox_se_grad_ws"]


def test_other_threads_run_while_a_launch_waits(gpu, tmp_path):
    """The operators bound to a library whose launches take 0.2 s (as they do when a queue is full) and do nothing: another
    thread, which wakes up every 2 ms, must go on meanwhile.  Nothing runs on the GPU."""
    lines = ["#include <time.h>"]
    for name in _abi.SIGNATURES:
        if name in WAITING:
            lines.append(f"int {name}(void) {{ struct timespec t = {{0, 200000000}}; nanosleep(&t, 0); return 0; }}")
        else:
            lines.append(f"long {name}(void) {{ return {3 if name == 'svox_out_data_dim' else 0}; }}")
    (tmp_path / "slow.c").write_text("\n".join(lines) + "\n")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "slow.so"), str(tmp_path / "slow.c")], check=True)
    tree = svox.N3Tree(data_format="RGBA", device=gpu)
    spec, opt = tree._spec(), options(tree)
    rays = rays_spec(synth.sphere_rays(64, seed=1), gpu)
    grad, points = torch.zeros(64, 3, device=gpu), torch.rand(64, 3, device=gpu)
    calls = [lambda: C.query_vertical(spec, points), lambda: C.query_vertical_backward(spec, points, torch.zeros(64, 4, device=gpu)),
             lambda: C.volume_render(spec, rays, opt), lambda: C.volume_render_backward(spec, rays, opt, grad, workspace=False),
             lambda: C.se_grad(spec, rays, grad, opt, workspace=False)]
    ticks, done = [0], threading.Event()

    def tick():
        while not done.is_set():
            ticks[0] += 1
            time.sleep(0.002)

    shim = C._shim()
    other = threading.Thread(target=tick)
    try:
        shim.init(str(tmp_path / "slow.so"))
        other.start()
        for call in calls:
            before = ticks[0]
            call()
            assert ticks[0] - before >= 20
    finally:
        done.set()
        shim.init(_abi.LIB_PATH)
        if other.ident:
            other.join()
