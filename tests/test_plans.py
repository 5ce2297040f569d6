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
    out, t, r = (C.c_int * 3)(), C.c_double(), C.c_double()
    lib.flash_plan_c(T, nq, nkv, pos0, int(bf16), cu, C.c_int64(room), out, C.byref(t), C.byref(r))
    return out[0], out[1], out[2], t.value, r.value


def test_key_ranges_fit_the_room_and_cover_the_keys(lib):
    rng = random.Random(7)
    for _ in range(3000):
        nq, nkv = rng.choice([(16, 2), (8, 2), (4, 1), (2, 1), (6, 2), (4, 4), (16, 1)])
        T, pos0, bf16 = int(2 ** rng.uniform(0, 12)), rng.choice([0, int(2 ** rng.uniform(5, 17))]), rng.random() < 0.5
        rooms = sorted(rng.sample(range(FULL + 1), 3)) + [FULL]
        before = None
        for room in [0] + rooms:
            piece, pieces, slots, t, _ = flash(lib, T, nq, nkv, pos0, bf16, room)
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
            _, _, slots, t, _ = flash(lib, T, nq, 2, pos0, bf16)
            half = flash(lib, T, nq, 2, pos0, bf16, FULL // 2)[3]
            assert half <= 1.3 * t, (T, pos0)
            if slots > FULL // 2:
                dropped = max(dropped, flash(lib, T, nq, 2, pos0, bf16, 0)[3] / t)
    assert dropped > 1.5


def image_floats(nkv, pos0, T):
    return nkv * -(-(pos0 + T) // 32) * 32 * 768  # 3 KB per position and head


def room(lib, T, nq, nkv, pos0, bf16, floats, cu=256):
    out, t = (C.c_int * 4)(), C.c_double()
    lib.attn_room_c(T, nq, nkv, pos0, int(bf16), cu, C.c_int64(floats), out, C.byref(t))
    return out[0], out[3], t.value


def test_image_and_partial_outputs_share_the_room(lib):
    """Both where both fit; the image where it fits unless cutting without it is expected to gain
    more; never past the room; nothing of it for a bf16 cache."""
    rng = random.Random(11)
    for _ in range(2000):
        nq, nkv = rng.choice([(16, 2), (8, 2), (4, 1), (2, 1), (4, 4)])
        T, pos0 = int(2 ** rng.uniform(0, 12)), rng.choice([0, int(2 ** rng.uniform(5, 16))])
        img = image_floats(nkv, pos0, T)
        _, _, slots, _, t = flash(lib, T, nq, nkv, pos0, False)
        assert room(lib, T, nq, nkv, pos0, False, img + slots * 4128) == (1, slots, t)
        assert room(lib, T, nq, nkv, pos0, True, 1 << 40)[:2] == (0, flash(lib, T, nq, nkv, pos0, True)[2])
        floats = int(rng.uniform(0, 1.2) * (img + slots * 4128))
        image, used, got = room(lib, T, nq, nkv, pos0, False, floats)
        assert image * img + used * 4128 <= floats
        alone = flash(lib, T, nq, nkv, pos0, False, floats // 4128)[4]
        beside = flash(lib, T, nq, nkv, pos0, False, max(0, floats - img) // 4128)
        gain = 1.35 if not beside[1] else 1.15 if -(-T * (nq // nkv) // 128) >= 8 else 1.0
        assert got == (beside[4] if image else alone)
        assert image == (img <= floats and beside[4] <= gain * alone)


def test_image_is_kept_beside_a_smaller_cut(lib):
    """16 / 2 heads, 54.6M floats less the query rows (the prompt arena's of 4096-token blocks of
    the 2B shape): turns for which both do not fit keep the image with a smaller cut where that
    measured faster, and leave it where it did not."""
    for T, pos0, keep in ((520, 18000, 1), (700, 16000, 1), (1200, 20000, 1), (700, 20000, 0), (520, 16000, 0)):
        floats = 54_600_000 - 16 * T * 256
        assert image_floats(2, pos0, T) + 4128 * flash(lib, T, 16, 2, pos0, False)[2] > floats
        image, slots, _ = room(lib, T, 16, 2, pos0, False, floats)
        assert image == keep and slots


def test_share_of_a_kept_workspace(lib):
    """Nothing where nothing is cut, enough for every cut of a shorter block at an earlier position
    up to half of the most, and never less for more tokens or positions."""
    share = lambda T, nq, nkv, b, ctx: lib.share_slots_c(T, nq, nkv, int(b), C.c_int64(ctx))  # noqa: E731
    rng = random.Random(5)
    for _ in range(1500):
        nq, nkv = rng.choice([(16, 2), (8, 2), (4, 1), (2, 1), (6, 2)])
        T, ctx, bf16 = int(2 ** rng.uniform(0, 13)), int(2 ** rng.uniform(5, 18)), rng.random() < 0.5
        n = share(T, nq, nkv, bf16, ctx)
        assert 0 <= n <= FULL // 2 and (n == 0) == (ctx <= 2048)
        assert n <= share(T + rng.randint(0, 64), nq, nkv, bf16, ctx + rng.randint(0, 5000))
        t = rng.randint(1, T)
        if t <= ctx:
            assert flash(lib, t, nq, nkv, rng.randint(0, ctx - t), bf16, FULL // 2)[2] <= n


# ----------------------------------------------------------------------- few-token GEMM
def small(lib, M, N, K, path, swiglu=False, cu=256):
    out = (C.c_int * 5)()
    return list(out) if lib.gemm_small_plan_c(M, N, K, int(swiglu), path, cu, out) else None


def test_few_token_gemm_plans(lib):
    """Every plan's tiles cover the product and hold no more than their form; its column tiles are
    within what a caller sets aside for their row maxima, on any number of compute units."""
    rng = random.Random(2)
    for _ in range(20000):
        swiglu = rng.random() < 0.5
        M, N, K = int(2 ** rng.uniform(0, 10.2)), int(2 ** rng.uniform(1, 15)), 8 * int(2 ** rng.uniform(0, 11))
        N += N % 2 if swiglu else 0
        cu = rng.choice([1, 7, 32, 64, 128, 256, 256, 256, 304, 512, 1024])
        p = small(lib, M, N, K, rng.randrange(3), swiglu, cu)
        if p is None:
            continue
        mr, nr, rt, ct, unit = p
        units, blocks = -(-N // unit), -(-M // 16)
        assert M <= 1024 and 1 <= ct <= units and 1 <= rt <= blocks
        assert unit % 2 == 0 or not swiglu
        assert -(-units // ct) * unit <= 16 * nr and -(-blocks // rt) <= mr
        assert ct <= lib.gemm_small_max_parts_c(N)


def test_the_tile_tests_reach_every_form(lib):
    from test_gpu_gemm_few_tokens_tiles import SIZES
    for f16, forms in SIZES.items():
        assert len(forms) == 12
        for form, sizes in forms.items():
            for s in sizes:
                assert tuple(small(lib, *s, path=int(f16))[:2]) == form, s
    assert small(lib, 1025, 1024, 2048, 0) is None


def test_shallow_products_with_the_fp16_split_leave_close_calls_to_the_tiles(lib):
    for M, N, K in ((256, 7168, 1024), (384, 5120, 1024), (300, 6144, 1024)):
        assert small(lib, M, N, K, 1) is None
    assert small(lib, 192, 5120, 1024, 1) and small(lib, 900, 2048, 2048, 1)
