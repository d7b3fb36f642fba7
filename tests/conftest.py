import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.dirname(os.path.abspath(__file__))
for p in (HERE, os.path.join(ROOT, "rils-rols_amd"), ROOT):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device); run with -m gpu")


def gpu_available():
    try:
        import torch  # noqa: F401  device count only; does not initialise HIP contexts
        return torch.cuda.device_count() > 0
    except Exception:
        return False


@pytest.fixture(scope="session")
def ctx():
    import capi
    c = capi.Context(0)
    yield c
    c.close()


OPTIONS = ("slab_budget_mb", "fp64_eval_rows", "fp64_eval_form", "fp32_rows", "fp32_chunk_rows", "fp32_streams",
           "host_threads", "phase_timing", "graph")


@pytest.fixture(autouse=True)
def _options_put_back(request):
    """Every test that uses the shared context finds it at its default options
    (four FP64 rows a thread, bucket streams by size), whatever the tests
    before it set or put back."""
    if "ctx" not in request.fixturenames:
        yield
        return
    c = request.getfixturevalue("ctx")
    keep = [(k, c.get_option(k)) for k in OPTIONS]
    yield
    for k, v in keep:
        c.set_option(k, v)
