"""The prefill kernels' cutting rules (csrc/plans.hpp, built with g++): CPU only."""
import ctypes as C
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FULL = 8192  # most slots


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("plans") / "plans.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "qwen3.5-cpu-cpp_amd", "csrc"), "-o", so,
                    os.path.join(ROOT, "tests", "cpp", "plans.cpp")], check=True)
    return C.CDLL(so)


def flash(lib, T, nq, nkv, pos0, bf16, room=FULL, cu=256):
    out, t = (C.c_int * 3)(), C.c_double()
    lib.flash_plan_c(T, nq, nkv, pos0, int(bf16), cu, C.c_int64(room), out, C.byref(t))
    return out[0], out[1], out[2], t.value


def test_key_ranges_fit_the_room_and_cover_the_keys(lib):
    rng = random.Random(7)
    for _ in range(3000):
        nq, nkv = rng.choice([(16, 2), (8, 2), (4, 1), (2, 1), (6, 2), (4, 4), (16, 1)])
        T, pos0, bf16 = int(2 ** rng.uniform(0, 12)), rng.choice([0, int(2 ** rng.uniform(5, 17))]), rng.random() < 0.5
        rooms = sorted(rng.sample(range(FULL + 1), 3)) + [FULL]
        before = None
        for room in [0] + rooms:
            piece, pieces, slots, t = flash(lib, T, nq, nkv, pos0, bf16, room)
            waves = 4 if bf16 else 8
            blocks = -(-T * (nq // nkv) // (16 * waves)) * nkv
            tiles = (pos0 + T - 1) // 32 + 1
            assert slots <= room and pieces <= 128
            if pieces:
                assert pieces > 1 and tiles > 64 and slots == pieces * blocks * waves
                assert (pieces - 1) * piece < tiles <= pieces * piece
            if before is not None:  # more room is never expected to be slower
                assert t <= before
            before = t


@pytest.mark.parametrize("nq,bf16", [(16, False), (8, False), (16, True), (8, True)])
def test_less_room_still_cuts(lib, nq, bf16):
    """A turn onto a long context with half of the most room: by the rule's own estimate never
    more than 1.3 times the time of the cut that takes all of it (a plan that does not fit is
    not simply dropped: unsplit these take up to 2.9 times as long)."""
    dropped = 0.0
    for pos0 in (2100, 4000, 8000, 16000, 32000):
        for T in range(20, 2049, 20):
            _, _, slots, t = flash(lib, T, nq, 2, pos0, bf16)
            half = flash(lib, T, nq, 2, pos0, bf16, FULL // 2)[3]
            assert half <= 1.3 * t, (T, pos0)
            if slots > FULL // 2:
                dropped = max(dropped, flash(lib, T, nq, 2, pos0, bf16, 0)[3] / t)
    assert dropped > 1.5
