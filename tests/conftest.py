import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (ROCm GPU) and the built libattnnn.so")


@pytest.fixture(scope="session")
def tiny_cfg():
    from attention_nn_amd.config import GPTConfig
    # the reference's own tiny self-test config (model.py:290-291)
    return GPTConfig(vocab_size=512, num_layers=2, num_heads=4, model_dim=64, seq_len=32,
                     window=16, long_layers=(1,))


def _trace(fn, tries=3):
    import torch
    from torch.autograd import DeviceType
    from torch.profiler import ProfilerActivity, profile
    for _ in range(tries):
        torch.cuda.synchronize()
        with profile(activities=[ProfilerActivity.CUDA]) as prof:
            fn()
            torch.cuda.synchronize()
        events = list(prof.events())
        on_device = sum(e.device_type == DeviceType.CUDA for e in events)
        if on_device >= sum("LaunchKernel" in e.name for e in events):   # else some were dropped
            break
    return [e.name for e in events]


@pytest.fixture(scope="session")
def traced():
    """traced(fn): the names of the kernels and runtime calls of one fn(), which is
    run again (up to `tries` times) where the trace lost some.
    Skipped where the profiler sees no kernels (another tracer holds the device)."""
    import torch
    x = torch.zeros(1024, device="cuda")
    if not any("elementwise" in n for n in _trace(lambda: x.add_(1))):
        pytest.skip("no kernel trace on this machine")
    return _trace
