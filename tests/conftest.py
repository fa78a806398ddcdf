import ctypes
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(scope="session")
def oracle():
    from oracle import oracle as o

    o.lib()
    return o


@pytest.fixture(scope="session")
def rnb():
    """The shipped package bound to librnb_hip.so; GPU tests skip cleanly when no device opens,
    mirroring the reference's device tests (crates/rnb-backend/cuda/src/runtime/tests.rs:22831-22834)."""
    import runnburn_amd as pkg

    if not pkg.device_available():
        pytest.skip(f"no HIP device: {pkg.last_error()}")
    return pkg


@pytest.fixture(scope="session")
def host_plan():
    """Host-side planning functions of the library (C++ linkage, no device needed), by mangled name and signature."""
    import runnburn_amd as pkg

    def bind(symbol, restype, *argtypes):
        fn = getattr(pkg.lib(), symbol)
        fn.restype, fn.argtypes = restype, list(argtypes)
        return fn

    return bind


@pytest.fixture(scope="session")
def two_digit_route(host_plan):
    """pays(quant, weight address, rows, cols, tokens): whether a K-quant / an importance-quant shape takes the two-digit GEMM."""
    sig = (ctypes.c_bool, ctypes.c_uint32, ctypes.c_void_p, *[ctypes.c_size_t] * 3)
    k_quants = host_plan("_ZN3rnb16gemm_digits_paysEjPKhmmm", *sig)
    importance = host_plan("_ZN3rnb19gemm_iq_digits_paysEjPKhmmm", *sig)
    return lambda quant, *args: (importance if quant >= 16 else k_quants)(quant, *args)
