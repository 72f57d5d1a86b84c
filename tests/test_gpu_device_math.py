"""rcp_n, div_n and sqrt_n (cn_math.h) against the device's IEEE operators,
bit for bit, over the ranges they are stated for: every reciprocal and root,
and random quotients with the ends of the mantissas among them."""

import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NATIVE = Path(__file__).resolve().parent / "native"


@pytest.fixture(scope="module")
def device_math(ctx):
    library = NATIVE / "libdevice_math.so"
    if not library.exists():
        subprocess.run(["make", "-C", str(NATIVE)], check=True)
    lib = C.CDLL(str(library))
    lib.device_math_every.argtypes = [C.c_int, C.c_uint32, C.c_uint32, C.c_void_p]
    lib.device_math_quotients.argtypes = [C.c_uint64, C.c_uint64, C.c_void_p]
    return lib


def bits(x):
    return int(np.float32(x).view(np.uint32))


def check(status, out):
    assert status == 0
    assert out[0] == 0, f"{out[0]} differ, {out[1] >> 32:#010x} / {out[1] & 0xFFFFFFFF:#010x} among them"


@pytest.mark.parametrize("root,low,high", [
    (0, 2.0**-126, 2.0**125), (0, 0.0, 0.0), (0, np.inf, np.inf),
    (1, 2.0**-101, np.inf), (1, 0.0, 0.0)])
def test_every_reciprocal_and_root(device_math, root, low, high):
    print("root" if root else "reciprocal", low, high, flush=True)
    out = (C.c_uint64 * 2)()
    check(device_math.device_math_every(root, bits(low), bits(high), out), out)


@pytest.mark.parametrize("seed", [1, 2])
def test_random_quotients(device_math, seed):
    print("quotients", seed, flush=True)
    out = (C.c_uint64 * 2)()
    check(device_math.device_math_quotients(seed << 40, 1 << 31, out), out)
