"""The batched product's launch rules on the CPU, against measured times."""
import os
import subprocess

import pytest

from gemm_shapes import BF16_SHORT_DIRECT, INT8_KERNELS, Q4_K, Q5_K, Q6_K, Q8_0

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    exe = tmp_path_factory.mktemp("plan") / "gemm_plan"
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-Werror",
                        "-I", os.path.join(ROOT, "agention-infer_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "gemm_plan.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(lines):
        r = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=60)
        assert r.returncode == 0
        out = [[int(v) for v in line.split()] for line in r.stdout.splitlines()]
        assert len(out) == len(lines)
        return out
    return run


def units(k):
    return (k + 255) // 256


# bf16 calls: (dtype, rows, k, tokens, us on the short-batch kernel, us on the
# 160 x 256 one).
SHORT_TIMES = [
    (Q4_K, 4800, 256, 64, 10.8, 12.0), (Q4_K, 4800, 256, 97, 13.8, 12.1), (Q4_K, 9000, 256, 64, 10.6, 14.0),
    (Q6_K, 18944, 256, 128, 15.9, 15.1), (Q8_0, 9000, 256, 64, 10.6, 13.8), (Q5_K, 14336, 256, 128, 15.3, 15.0),
    (Q6_K, 1200, 256, 16, 9.0, 11.8), (Q6_K, 4800, 512, 128, 14.7, 18.4), (Q4_K, 18944, 512, 128, 15.5, 25.9),
    (Q4_K, 18944, 3584, 64, 28.2, 44.6), (Q4_K, 37888, 256, 32, 13.2, 12.1), (Q8_0, 37888, 256, 1, 13.8, 10.9),
    (Q8_0, 37888, 256, 128, 27.3, 15.0), (Q6_K, 37888, 512, 128, 28.1, 21.3), (Q4_K, 37888, 1024, 128, 28.4, 28.3),
    (Q6_K, 65536, 256, 64, 28.2, 24.3), (Q8_0, 65536, 512, 112, 40.1, 33.1), (Q8_0, 128256, 256, 96, 53.4, 42.0),
]


def test_quad_kernel_rule(ask):
    """A short batch takes the faster kernel, to within the estimates' error."""
    got = ask([f"quad {t} {r} {units(k)} {n}" for t, r, k, n, _, _ in SHORT_TIMES])
    for (t, r, k, n, short, direct), (_, quad) in zip(SHORT_TIMES, got):
        taken, other = (short, direct) if quad else (direct, short)
        assert taken <= 1.1 * other, f"dtype {t}, {r} x {k} at {n} tokens: takes {taken} us, the other {other}"


# Q6_K int8 calls: (rows, k, tokens, us on the 64 x 64 blocks, us on the
# 160-row ones with their K split).
Q6_TIMES = [
    (64, 256, 2, 8.2, 15.1), (133, 256, 200, 9.9, 16.0), (600, 256, 200, 11.0, 16.4), (2400, 256, 128, 10.9, 17.6),
    (4800, 256, 300, 13.8, 18.2), (9000, 256, 512, 26.6, 19.3), (14336, 256, 64, 10.9, 16.5),
    (18944, 256, 384, 33.8, 25.6), (133, 512, 2, 12.1, 14.7), (1200, 512, 512, 15.4, 20.0),
    (4800, 512, 200, 17.1, 23.3), (9000, 512, 384, 29.9, 24.1), (9000, 512, 700, 43.7, 31.8),
    (2400, 768, 700, 24.8, 32.6), (4800, 768, 300, 24.5, 31.4), (9000, 768, 700, 57.6, 42.5),
    (14336, 768, 200, 34.0, 31.9), (64, 1024, 2, 20.2, 15.8), (600, 1024, 16, 21.3, 16.4),
    (2400, 1024, 300, 23.7, 24.7), (4800, 1024, 300, 30.1, 32.5), (9000, 1024, 512, 54.9, 40.4),
    (9000, 1280, 300, 43.5, 46.7), (133, 2048, 64, 37.3, 17.3), (3584, 2048, 512, 53.6, 47.8),
    (3584, 3072, 64, 54.6, 28.3),
]


# bf16 calls on the short-batch kernel: (dtype, rows, k, tokens, us unsplit, us in
# 2 K splits).
SPLIT_TIMES = [
    (Q4_K, 3584, 1280, 128, 21.6, 18.2), (Q4_K, 4800, 1280, 96, 18.9, 16.9), (Q8_0, 3584, 2048, 128, 22.0, 18.4),
    (Q8_0, 4800, 2048, 96, 19.4, 16.9), (Q8_0, 9000, 2048, 48, 15.2, 14.9), (Q4_K, 14336, 2048, 48, 14.8, 15.9),
    (Q8_0, 14336, 2048, 96, 22.2, 23.6), (Q8_0, 14336, 2048, 128, 25.4, 27.6), (Q8_0, 14336, 1280, 128, 23.6, 25.9),
    (Q6_K, 37888, 3584, 48, 53.6, 55.5), (Q4_K, 37888, 3584, 96, 66.0, 67.6), (Q8_0, 65536, 3584, 64, 97.8, 103.7),
    (Q4_K, 14336, 2048, 96, 19.3, 22.4), (Q4_K, 14336, 2048, 128, 22.8, 26.4), (Q6_K, 65536, 3584, 128, 128.6, 136.7),
    (Q8_0, 65536, 3584, 128, 134.1, 142.9), (Q6_K, 37888, 4096, 64, 60.9, 64.2), (Q4_K, 37888, 4096, 128, 79.2, 81.4),
]


# (dtype, rows, k, tokens, us in 1, 2, ... splits): few tokens, where rounds of
# single quads are slower than their count tells.
SPLITS_TIMES = [
    (Q6_K, 9886, 8192, 3, [42.2, 27.8, 38.8, 30.9, 31.0, 41.9, 42.3, 31.5]),
    (Q8_0, 171, 12192, 25, [57.5, 34.0, 25.5, 21.9, 22.1, 18.5, 19.1, 19.4, 20.3, 20.4, 20.4, 17.4]),
    (Q6_K, 12071, 6912, 24, [40.1, 30.5, 41.5, 34.1, 43.7, 45.4, 36.3]),
    (Q6_K, 14976, 7680, 10, [42.2, 47.9, 39.4, 42.5, 42.2, 52.7, 51.7, 45.0]),
    (Q5_K, 12198, 6400, 21, [41.4, 30.9, 41.9, 34.1, 44.0, 44.9, 35.1]),
    (Q6_K, 14618, 7680, 3, [41.8, 48.0, 40.0, 43.0, 42.7, 52.3, 52.4, 45.4]),
    (Q6_K, 10396, 13056, 2, [64.1, 42.0, 56.2, 48.0, 40.9, 54.7, 43.7, 43.7, 48.2, 48.8, 49.1, 55.2, 46.4]),
    (Q8_0, 12266, 1152, 24, [15.4, 14.0]),
    (Q4_K, 14105, 2304, 9, [17.4, 16.0, 16.0]),
]


def test_quad_split_rule(ask):
    """A K split earns its reduction, its launch and the partial products'
    traffic that grows with tokens and rows, to within the estimate's error."""
    got = ask([f"quad {t} {r} {units(k)} {n}" for t, r, k, n, _, _ in SPLIT_TIMES])
    for (t, r, k, n, one, two), (ks,) in zip(SPLIT_TIMES, ((g[0],) for g in got)):
        assert {1: one, 2: two}[ks] <= 1.1 * min(one, two), f"dtype {t}, {r} x {k} at {n} tokens: {ks} splits"
    got = ask([f"quad {t} {r} {units(k)} {n}" for t, r, k, n, _ in SPLITS_TIMES])
    for (t, r, k, n, us), g in zip(SPLITS_TIMES, got):
        assert us[g[0] - 1] <= 1.05 * min(us), f"dtype {t}, {r} x {k} at {n} tokens: {g[0]} splits"


def test_q6_small_rule(ask):
    """The rule takes the faster of the two kernels wherever they differ by
    more than the estimates can tell."""
    got = ask([f"q8 {Q6_K} {r} {units(k)} {n}" for r, k, n, _, _ in Q6_TIMES])
    for (r, k, n, small, big), g in zip(Q6_TIMES, got):
        taken, other = (small, big) if g[0] else (big, small)
        assert taken <= 1.05 * other, f"{r} x {k} at {n} tokens: takes {taken} us, the other {other}"


def test_test_shapes_take_their_kernel(ask):
    got = ask([f"quad {t} {r} {units(k)} {n}" for t, r, k, n in BF16_SHORT_DIRECT])
    assert [g[1] for g in got] == [0] * len(got)
    got = ask([f"q8 {t} {r} {units(k)} {n}" for t, r, k, n, _ in INT8_KERNELS])
    for (t, r, k, n, kernel), g in zip(INT8_KERNELS, got):
        assert kernel == ("small" if g[0] else 128 * g[1]), f"dtype {t}, {r} x {k} at {n} tokens: {g}"


def test_q8_workspace_bound(ask):
    """The bound for batches of up to n tokens covers each of them."""
    shapes = [(t, r, u) for t in (Q4_K, Q6_K) for r, u in
              ((1, 1), (133, 2), (91, 4), (512, 14), (3584, 74), (18944, 14), (161, 6), (40000, 3))]
    for t, r, u in shapes:
        got = ask([f"q8 {t} {r} {u} {n}" for n in range(1, 700, 13)])
        bytes_ = [g[3] for g in got]
        for i, g in enumerate(got):
            assert max(bytes_[:i + 1]) <= g[4]


def test_room_tokens(ask):
    """A batch that grows token by token takes few workspaces, and the kept
    ones come to at most 3 times the last."""
    sizes = [g[0] for g in ask([f"room {n}" for n in range(1, 9000)])]
    assert all(n <= s <= max(256, 3 * n // 2 + 256) for n, s in enumerate(sizes, 1))
    steps = sorted(set(sizes))
    assert sizes == sorted(sizes) and len(steps) <= 12
    for i in range(1, len(steps)):
        assert sum(steps[:i]) <= 3 * steps[i]


def test_take_workspace(ask):
    """Room beyond a call's own bytes is taken where it can be had, and the
    call goes on without where not (and does not ask again each time)."""
    big = 1 << 60
    cases = {
        (0, big, 10, 50, 100): (1, 50, big, 1),   # room to be had
        (0, big, 10, 50, 20): (1, 10, 50, 2),     # only its own bytes
        (10, 50, 10, 50, 20): (1, 10, 50, 0),     # held, the room refused before
        (10, big, 10, 50, 20): (1, 10, 50, 1),    # held, the room refused now
        (10, 50, 10, 40, 45): (1, 40, 50, 1),     # less room than was refused
        (10, 50, 30, 60, 35): (1, 30, 50, 1),     # growth, room known to be refused
        (0, big, 10, 50, 5): (0, 0, 50, 2),       # not even that
        (60, big, 10, 50, 100): (1, 60, big, 0),  # held
    }
    got = ask(["take " + " ".join(map(str, c)) for c in cases])
    assert [tuple(g) for g in got] == list(cases.values())
