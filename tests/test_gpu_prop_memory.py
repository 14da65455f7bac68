"""The proposal field where the memory does not hold the staged features: one kernel, whose values
are the same to the bit (as test_gpu_prop_levels states)."""
import pytest
import torch

from neural3dstrokes_amd import _lib, propfield


@pytest.mark.gpu
def test_without_memory_for_the_stage(dev):
    torch.manual_seed(0)
    m = propfield.PropDensityField().to(dev).eval().requires_grad_(False)
    m.encoder.embeddings.data.uniform_(-0.3, 0.3)
    n = 1 << 22
    x = torch.randn(n, 3, device=dev)
    need = _lib.lib().n3ds_prop_field_workspace_bytes(n, 10, 1, m.encoder.embeddings.shape[0], 0)
    assert need >= 160 << 20
    with torch.no_grad():
        want = m(x)['density'].clone()
        torch.cuda.empty_cache()
        total = torch.cuda.get_device_properties(dev).total_memory
        # the outputs take 28 bytes a point, 112 MiB
        limit = torch.cuda.memory_reserved() + (150 << 20)
        try:
            torch.cuda.set_per_process_memory_fraction(limit / total)
            got = m(x)['density']
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got, want)
