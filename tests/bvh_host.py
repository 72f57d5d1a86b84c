"""The host BVH builder for CPU tests: cn_bvh.cpp and a C call around it
(native/bvh_host.cpp), compiled with the flags the library's host files use,
and the scenes whose trees come near the builder's limits."""

import ctypes as C
import functools
import subprocess
import tempfile
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parents[1]
STACK_MAX = 128  # cn_launch.h: the traversal stack's entries


@functools.lru_cache(maxsize=None)
def _library():
    source = ROOT / "cenote_amd" / "csrc"
    out = Path(tempfile.mkdtemp(prefix="bvh_host_")) / "libbvh_host.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-fno-fast-math",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{source}", str(source / "cn_bvh.cpp"),
                    str(ROOT / "tests" / "native" / "bvh_host.cpp"), "-pthread", "-o", str(out)], check=True)
    lib = C.CDLL(str(out))
    lib.bvh_host_build.argtypes = [C.c_void_p] + [C.c_uint32] * 4 + [C.POINTER(C.c_uint32)] * 4 + [
        C.c_char_p, C.c_size_t]
    return lib


def build(corners, max_stack=STACK_MAX, nodes4=1 << 26, nodes8=1 << 25):
    """The trees over (n, 3, 3) corners: their node counts and depths, and
    the refusal's text (empty when built)."""
    corners = np.ascontiguousarray(corners, np.float32)
    values = [C.c_uint32() for _ in range(4)]
    error = C.create_string_buffer(256)
    _library().bvh_host_build(corners.ctypes.data_as(C.c_void_p), len(corners), max_stack, nodes4,
                              nodes8, *[C.byref(v) for v in values], error, len(error))
    return dict(zip(("nodes4", "depth4", "nodes8", "depth8"), (v.value for v in values))), error.value.decode()


def chain(levels, cluster=6):
    """Clusters of well-separated triangles, each a quarter of the size of the
    one before: a deep tree, and with some lengths a level or two deeper by the
    usual rules than by the coarse ones."""
    rng = np.random.default_rng(1)
    scale = np.ldexp(1.0, 56 - 2 * np.arange(levels)).repeat(cluster)[:, None, None]
    n = levels * cluster
    at = np.concatenate([rng.uniform(0.9, 1.0, (n, 1, 1)), rng.uniform(0, 1, (n, 1, 2))], axis=2)
    shape = np.array([[0, 0, 0], [1e-3, 0, 0], [0, 1e-3, 1e-3]])
    return ((at + shape) * scale).astype(np.float32)


def lattice(side):
    """Small triangles far apart: every one of them a leaf of its own."""
    at = np.stack(np.meshgrid(*[np.arange(side)] * 3, indexing="ij"), axis=-1).reshape(-1, 1, 3)
    return (at + np.array([[0, 0, 0], [1e-3, 0, 0], [0, 1e-3, 1e-3]])).astype(np.float32)
