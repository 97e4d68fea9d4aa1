"""The brick kernel's bounds of rows and samples (bound_slice and clip_row of
rexlib_amd/csrc/section_bounds.hpp), compiled for the CPU and compared with a
walk over every sample of a slice: no sample whose first tap lies in a brick is
dropped, for both copies of a slice, every window, brick shape, extent and last
shell; no sample that the slice does not insert is kept (its prepared value is
not written); and few rows without a sample are kept. The reciprocals, which
are approximate on the device, are off by up to two units in the last place
either way; the functions are built with and without fused multiply-adds."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from rexlib_amd import tune

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "rexlib_amd", "csrc")
COMPILER = next((c for c in ("/opt/rocm/bin/amdclang++", "/opt/rocm/llvm/bin/clang++", shutil.which("clang++"))
                 if c and os.path.exists(c)), None)
# Half-width and layout taps: nearest, trilinear, Kaiser-Bessel of 3 and 4 taps.
WINDOWS = [(0.5, 1), (1.0, 2), (1.2, 4), (1.5, 4), (2.0, 4)]


@pytest.fixture(scope="module", params=["fused", "unfused"])
def check(request, tmp_path_factory):
    path = str(tmp_path_factory.mktemp("bounds") / "check.so")
    flags = ["-mfma", "-ffp-contract=fast"] if request.param == "fused" else ["-ffp-contract=off"]
    subprocess.run([COMPILER, "-std=c++17", "-O2", "-fPIC", "-shared", *flags, "-I", CSRC, "-o", path,
                    os.path.join(HERE, "section_bounds_check.cpp")], check=True)
    function = ctypes.CDLL(path).section_bounds_check
    p = ctypes.c_void_p
    function.argtypes = [ctypes.c_int, p, p, ctypes.c_int, ctypes.c_int, ctypes.c_float, p, p, ctypes.c_int, p]
    function.restype = None

    def run(n, frame, last_shell, window, low, extent, ulps, out):
        x, y = frame[0].astype(np.float32), np.ascontiguousarray(frame[1], np.float64)
        low, extent = np.asarray(low, np.int32), np.asarray(extent, np.int32)
        function(n, x.ctypes.data, y.ctypes.data, last_shell, window[1], window[0], low.ctypes.data, extent.ctypes.data,
                 ulps, out.ctypes.data)

    return run


def rotation(rng):
    q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    return q


def frame_of(kind, rng):
    """Steps of k_x and k_y for N = n: rotations; planes along the lattice's
    axes (zero steps and zero normals); matrices of any shape, as the insertion
    accepts; axes a small angle apart."""
    if kind == "rotation":
        return rotation(rng)[:2]
    if kind == "axes":
        return (np.eye(3)[rng.permutation(3)] * rng.choice([-1.0, 1.0], 3)[:, None])[:2]
    if kind == "any":
        return rng.uniform(-1, 1, (2, 3))
    if kind == "one axis":
        # k_x runs along an axis, k_y nearly so.
        f = np.eye(3)[rng.permutation(3)][:2]
        f[1] = f[0] + rng.uniform(-1, 1, 3) * 10.0 ** rng.uniform(-6, 0)
        return f
    r = rotation(rng)
    return np.stack([r[0], r[0] + r[1] * 10.0 ** rng.uniform(-3, 0)])


def transforms_as_float32(frame):
    return frame.astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("kind", ["rotation", "axes", "any", "one axis", "near"])
@pytest.mark.parametrize("n", [5, 8, 63, 128, 255])
def test_no_sample_of_a_brick_is_dropped(check, kind, n):
    rng = np.random.default_rng(n)
    out = np.zeros(5, np.int64)
    for case in range(400):
        scale = rng.choice([1.0, 2.0, 0.7, rng.uniform(0.3, 8.0)])
        frame = transforms_as_float32(frame_of(kind, rng)) * scale
        last = int(rng.choice([n // 2, n // 2, n // 3, 1, 0]))
        window = WINDOWS[rng.integers(len(WINDOWS))]
        extent = tune.SHAPES[rng.integers(len(tune.SHAPES))]
        # A brick around some sample of the slice.
        centre = rng.uniform(-last, last, 2) @ frame * rng.choice([-1, 1])
        low = np.floor(centre - np.array(extent) * rng.uniform(0, 1, 3)).astype(int)
        before = out.copy()
        check(n, frame, last, window, low, extent, int(rng.integers(-2, 3)), out)
        assert out[1] == before[1], (case, frame, last, window, low, extent)
        assert out[4] == before[4], (case, frame, last, window, low, extent)
    assert out[0] > 400
    if kind == "rotation" and n > 100:
        # At most one row in three holds no sample (those of few samples per
        # voxel among them).
        assert out[2] < 1.5 * out[3]


# The longest extents that are not written past the last shell (4,095), and the
# first whose shells are found without the rounded square root's correction.
@pytest.mark.parametrize("n", [719, 721, 2048, 4095])
def test_large_extents(check, n):
    rng = np.random.default_rng(n)
    out = np.zeros(5, np.int64)
    for case in range(12):
        frame = transforms_as_float32(rotation(rng)[:2])
        last = int(rng.choice([n // 2, n // 2 - 1, n // 3]))
        centre = rng.uniform(-last, last, 2) / 1.5 @ frame
        check(n, frame, last, WINDOWS[case % len(WINDOWS)], np.floor(centre).astype(int) - 4, (16, 16, 8), 0, out)
    assert out[0] > 12 and out[1] == 0 and out[4] == 0


# Rows along the lattice's x axis in a brick at its edge: the clipped rows end at
# the shell itself.
@pytest.mark.parametrize("n", [255, 256, 1024, 4094, 4095])
def test_rows_end_at_the_last_shell(check, n):
    out = np.zeros(5, np.int64)
    frame = np.array([[1.0, 0.0, 0.0], [0.0, 1.0, 0.0]])
    for last in (n // 2, n // 2 - 1, n // 2 - 7):
        check(n, frame, last, (1.0, 2), (last - 12, -n // 2, -4), (40, n + 2, 8), 0, out)
        check(n, frame, last, (1.0, 2), (0, -n // 2, -4), (n, n + 2, 8), 0, out)
    assert out[0] > 100 and out[1] == 0 and out[4] == 0
