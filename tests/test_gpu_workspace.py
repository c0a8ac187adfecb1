"""How much memory torch's allocator holds and no tensor has, as the size of a workspace goes by it."""
import pytest
import torch

import svox_amd.csrc as C

pytestmark = pytest.mark.gpu


def test_cached_bytes_are_the_allocators(gpu):
    def same():
        return C._shim().cached_bytes(gpu.index or 0) == torch.cuda.memory_reserved(gpu) - torch.cuda.memory_allocated(gpu)

    torch.cuda.empty_cache()
    assert same()
    held = torch.empty(100 << 20, dtype=torch.uint8, device=gpu)
    small = torch.empty(1000, dtype=torch.uint8, device=gpu)
    assert same()
    del held
    assert C._shim().cached_bytes(gpu.index or 0) >= 100 << 20 and same()
    del small
    torch.cuda.empty_cache()
    assert same()
