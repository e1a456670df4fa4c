import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "burn-rocket_amd")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")


@pytest.fixture(params=["few-rows", "128-rows"])
def attn_route(request, monkeypatch):
    """Shapes of few query rows on the kernel the library picks for them, and on the 128-row kernel
    (with its transposed V) that larger ones take."""
    if request.param == "128-rows":
        monkeypatch.setenv("RK_ATTN_FEW", "0")


@pytest.fixture(scope="session")
def orc():
    import oracle
    oracle.lib()
    return oracle


@pytest.fixture(scope="session")
def rk():
    """The library, initialised on device 0 (GPU tests only)."""
    import burn_rocket
    burn_rocket.init(0)
    return burn_rocket
