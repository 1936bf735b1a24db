"""GPU parity for the batched prefill GEMM (gq_gemm) against CPU references.

Both modes change the operands' precision by definition, so each is
compared against a CPU matmul of the *same* operands (tolerance
max|err| <= 1e-4 * max|y_ref|, fp64 reference):
  * GQ_GEMM_BF16: W = bf16(dequant(W)) (round to nearest even of the
    bit-exact fp32 dequant), X = bf16(X).
  * GQ_GEMM_INT8: W = dequant(W) exactly, X = per-32 Q8 pack of X
    (KvDtype::Q8_0::pack, src/model/mod.rs:574-583), i.e. q * f16(scale).
The distance to the fp32 CPU path (WeightMap::matmul_batch_into,
src/model/mod.rs:414-464) is also checked, with a tolerance that reflects
the operand rounding (bf16: 2^-9 relative per operand).
"""
import sys

import numpy as np
import pytest

import gq_synth as syn
from gemm_shapes import BF16_SHORT_DIRECT, INT8_KERNELS

pytestmark = pytest.mark.gpu

Q4_K = 12
TOL = 1e-4


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def bf16_round(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32).astype(np.uint64)
    r = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16
    return r.astype(np.uint32).view(np.float32)


def run(backend, orc, rows, k, n, mode, seed, dtype=Q4_K):
    import torch
    import gq
    w = syn.make_blocks(dtype, rows, k, seed=seed)
    X = syn.make_x(k, seed=seed + 1, batch=n)
    h = backend.upload_weight(dtype, w, k, rows)
    Y = h.launch_only_batch(torch.from_numpy(X).cuda(), mode=mode)
    torch.cuda.synchronize()
    Wf = orc.dequant(dtype, w.reshape(-1), rows * k).reshape(rows, k) if k % 256 == 0 else \
        orc.dequant_rows(dtype, w, k)
    return w, X, Wf, Y.cpu().numpy()


def check(y, ref, what, tol=TOL):
    err = float(np.max(np.abs(y.astype(np.float64) - ref)))
    bound = tol * float(np.max(np.abs(ref)))
    say(f"{what}: max|err| {err:.3g} bound {bound:.3g}")
    assert err <= bound, f"{what}: max|err| {err:.3g} > {bound:.3g}"


SHAPES = [(331, 512, 37), (1024, 3584, 64), (160, 256, 256), (7, 300, 5), (2000, 1024, 300)]
Q6_K = 14
# Q6_K (the ffn_down / attn_v type of Q4_K_M files): narrow and wide token
# tiles, K splits (few row tiles), a partial last unit.
Q6_SHAPES = [(331, 512, 37), (512, 2048, 300), (100, 768, 20), (3584, 2048, 512), (40, 300, 3)]


@pytest.mark.parametrize("rows,k,n", Q6_SHAPES)
def test_gemm_bf16_q6k(backend, orc, rows, k, n):
    import gq
    say(f"gemm bf16 Q6_K rows={rows} k={k} n={n}")
    w, X, Wf, Y = run(backend, orc, rows, k, n, gq.GQ_GEMM_BF16, seed=rows + 7 * k, dtype=Q6_K)
    ref = bf16_round(X).astype(np.float64) @ bf16_round(Wf).astype(np.float64).T
    check(Y, ref, "bf16 Q6_K vs same-operand fp64")


@pytest.mark.parametrize("rows,k,n", SHAPES)
def test_gemm_bf16(backend, orc, rows, k, n):
    import gq
    say(f"gemm bf16 rows={rows} k={k} n={n}")
    w, X, Wf, Y = run(backend, orc, rows, k, n, gq.GQ_GEMM_BF16, seed=rows + k)
    ref = bf16_round(X).astype(np.float64) @ bf16_round(Wf).astype(np.float64).T
    check(Y, ref, "bf16 vs same-operand fp64")
    ref32 = orc.matmul_batch_into(Q4_K, w, X, rows)
    check(Y, ref32, "bf16 vs fp32 CPU path", tol=1e-2)


@pytest.mark.parametrize("dtype,rows,k,n", [
    (Q4_K, 113, 5120, 1), (Q6_K, 97, 1280, 16), (13, 225, 2304, 17), (8, 111, 4128, 33), (Q4_K, 1, 256, 50),
    (Q6_K, 500, 3072, 81), (13, 112, 1024, 96), (8, 130, 1056, 97), (Q4_K, 3001, 1792, 128), (Q6_K, 16, 9728, 128)])
def test_gemm_bf16_short(backend, orc, dtype, rows, k, n):
    """Batches of up to 128 tokens: every number of token tiles, row tiles of
    112 with remainders, last quads of 1 to 4 units, K split or not."""
    import gq
    say(f"gemm bf16 short dtype={dtype} rows={rows} k={k} n={n}")
    w, X, Wf, Y = run(backend, orc, rows, k, n, gq.GQ_GEMM_BF16, seed=rows + 3 * k + n, dtype=dtype)
    ref = bf16_round(X).astype(np.float64) @ bf16_round(Wf).astype(np.float64).T
    check(Y, ref, "bf16 vs same-operand fp64")


@pytest.mark.parametrize("dtype,rows,k,n", BF16_SHORT_DIRECT)
def test_gemm_bf16_short_direct(backend, orc, dtype, rows, k, n):
    """Batches of up to 128 tokens that take the 160 x 256 kernel."""
    import gq
    say(f"gemm bf16 short direct dtype={dtype} rows={rows} k={k} n={n}")
    w, X, Wf, Y = run(backend, orc, rows, k, n, gq.GQ_GEMM_BF16, seed=rows + 3 * k + n, dtype=dtype)
    ref = bf16_round(X).astype(np.float64) @ bf16_round(Wf).astype(np.float64).T
    check(Y, ref, "bf16 vs same-operand fp64")


def test_gemm_bf16_short_experts(backend, orc):
    """Stacked experts of 24 rows (the wave-tiled layout) in a short batch."""
    import gq
    import torch
    E, f, k, n = 3, 24, 512, 19
    w = syn.make_blocks(Q4_K, E * f, k, seed=9)
    X = syn.make_x(k, seed=10, batch=n)
    h = backend.upload_experts(Q4_K, w, k, f, E)
    Y = h.launch_only_batch(torch.from_numpy(X).cuda(), mode=gq.GQ_GEMM_BF16).cpu().numpy()
    Wf = orc.dequant(Q4_K, w.reshape(-1), E * f * k).reshape(E * f, k)
    check(Y, bf16_round(X).astype(np.float64) @ bf16_round(Wf).astype(np.float64).T, "experts vs same-operand fp64")


@pytest.mark.parametrize("dtype,rows,k,n", [(Q4_K,) + sh for sh in SHAPES] + [(Q6_K,) + sh for sh in Q6_SHAPES]
                         + [(Q6_K, 3584, 18944, 512)])
def test_gemm_int8(backend, orc, dtype, rows, k, n):
    """GQ_GEMM_INT8 for Q4_K and Q6_K weights (Q4_K_M files keep ffn_down and
    attn_v in Q6_K; 3584 x 18944 is the 7B down projection) against the
    same-operand fp64 product and the fp32 CPU path."""
    import gq
    say(f"gemm int8 dtype={dtype} rows={rows} k={k} n={n}")
    w, X, Wf, Y = run(backend, orc, rows, k, n, gq.GQ_GEMM_INT8, seed=rows + k + 1, dtype=dtype)
    kp = (k + 31) // 32 * 32
    Xq = np.zeros((n, k), np.float64)
    for t in range(n):
        sc, q = orc.quantize_q8_32(X[t])
        s = np.repeat(sc.view(np.float16).astype(np.float64), 32)[:kp]
        Xq[t] = (q.astype(np.float64) * s[: q.size])[:k]
    ref = Xq @ Wf.astype(np.float64).T
    check(Y, ref, "int8 vs same-operand fp64")
    sub = np.arange(0, n, max(1, n // 16))
    ref32 = orc.matmul_batch_into(dtype, w, X[sub], rows)
    check(Y[sub], ref32, "int8 vs fp32 CPU path", tol=3e-2)


@pytest.mark.parametrize("dtype", [Q4_K, Q6_K])
@pytest.mark.parametrize("rows,k,n", [(1, 256, 1), (161, 1536, 129), (321, 2560, 257), (2400, 768, 384), (159, 5000, 128)])
def test_gemm_int8_tiles(backend, orc, dtype, rows, k, n):
    """The 128-token tile (both are in test_gemm_int8_kernels), one row past a
    tile and one short of it, K splits of uneven units, a ragged last unit;
    Q6_K scales at both ends of int8, where sc (q - 32) passes 11 bits, and
    activations whose blocks differ by 2^16 in one unit.  In every third token
    only the small block is left, and errors count against the token's own
    results (bound: test_gemm_int8_kernels)."""
    import gq
    import torch
    say(f"gemm int8 tiles dtype={dtype} rows={rows} k={k} n={n}")
    rng = np.random.default_rng(rows + k + n)
    w = syn.make_blocks(dtype, rows, k, seed=rows + n)
    if dtype == Q6_K:
        b = w.reshape(rows, -1, 210)
        b[..., 192:208] = rng.integers(-128, 128, b[..., 192:208].shape, dtype=np.int8).view(np.uint8)
    X = syn.make_x(k, seed=n, batch=n)
    X[:, :32] *= np.float32(2.0 ** -8)  # (scales of 1e-4 and 5, both normal in f16)
    X[:, 32:64] *= np.float32(2.0 ** 8)
    X[::3, 32:] = 0
    h = backend.upload_weight(dtype, w, k, rows)
    Y = h.launch_only_batch(torch.from_numpy(X).cuda(), mode=gq.GQ_GEMM_INT8).cpu().numpy()
    check_tokens(Y, int8_ref(orc, dtype, w, X), 1e-6 if rows > 1 else 1e-5)


def int8_ref(orc, dtype, w, X):
    """The int8 mode's product in float64: exact dequant times the Q8 pack."""
    n, k = X.shape
    Xq = np.zeros((n, k), np.float64)
    for t in range(n):
        sc, q = orc.quantize_q8_32(X[t])
        Xq[t] = q.astype(np.float64) * np.repeat(sc.view(np.float16).astype(np.float64), 32)[:k]
    return Xq @ orc.dequant_rows(dtype, w, k).astype(np.float64).T


def check_tokens(Y, ref, tol):
    """Every token's error against the size of its own results (2-norms)."""
    assert np.all(np.isfinite(Y))
    err = np.sqrt(np.mean((Y - ref) ** 2, axis=1)) / np.sqrt(np.mean(ref ** 2, axis=1) + 1e-300)
    say(f"  worst token {err.max():.3g}, bound {tol:.3g}")
    assert err.max() <= tol


@pytest.mark.parametrize("dtype,rows,k,n,kernel", INT8_KERNELS)
def test_gemm_int8_kernels(backend, orc, dtype, rows, k, n, kernel):
    """Each kernel of the int8 mode at the edges of its tiles.  Every integer
    in it is exact, so per token only the roundings of 8 sums per unit and one
    or two per unit of the result, and the reference's f32 weights, are left: up
    to 2^-24 each of partial sums below the result's size, about 1.5e-7 together
    for 20 units, bounded here by 1e-6."""
    import gq
    import torch
    say(f"gemm int8 {kernel} dtype={dtype} rows={rows} k={k} n={n}")
    rng = np.random.default_rng(rows + k + n)
    w = syn.make_blocks(dtype, rows, k, seed=rows + n)
    if dtype == Q6_K:  # scales over all of int8
        b = w.reshape(rows, -1, 210)
        b[..., 192:208] = rng.integers(-128, 128, b[..., 192:208].shape, dtype=np.int8).view(np.uint8)
    X = syn.make_x(k, seed=n, batch=n)
    ref = int8_ref(orc, dtype, w, X)
    h = backend.upload_weight(dtype, w, k, rows)
    for off in (0, 1):  # X aligned, and to 4 bytes only
        buf = torch.zeros(n * k + 1, device="cuda")
        buf[off:off + n * k] = torch.from_numpy(X).cuda().view(-1)
        Y = h.launch_only_batch(buf[off:off + n * k].view(n, k), mode=gq.GQ_GEMM_INT8).cpu().numpy()
        check_tokens(Y, ref, 1e-6 if rows > 1 else 1e-5)  # (one row: it may be small beside its terms)


@pytest.mark.parametrize("rows,k,n", [(320, 1024, 130), (18944, 250, 260)])
def test_gemm_int8_min_term(backend, orc, rows, k, n):
    """Q4_K results that are all min term: xs sum(q) has 23 bits and goes through
    the MFMA in three bf16.  What is left is f32 rounding (as in
    test_gemm_int8_kernels, below 5e-7); a product with two of the three is
    further off than that."""
    import gq
    import torch
    say(f"gemm int8 min term rows={rows} k={k} n={n}")
    w = syn.make_blocks(Q4_K, rows, k, seed=91)
    b = w.reshape(rows, -1, 144)
    b[..., 0:2] = np.zeros(1, np.float16).view(np.uint8)  # d = 0
    X = syn.make_x(k, seed=92, batch=n)
    ref = int8_ref(orc, Q4_K, w, X)
    xs, m = np.zeros((n, (k + 31) // 32)), np.zeros((rows, (k + 31) // 32))
    for t in range(n):
        sc, q = orc.quantize_q8_32(X[t])
        q = np.pad(q.astype(np.float64), (0, 32 * xs.shape[1] - q.size)).reshape(-1, 32)
        xs[t] = sc.view(np.float16).astype(np.float64)[:xs.shape[1]] * q.sum(1)
    m = -orc.dequant_rows(Q4_K, w, k).astype(np.float64)[:, ::32]
    x1 = bf16_round(xs)
    two = x1.astype(np.float64) + bf16_round(xs - x1)
    size = np.sqrt(np.mean(ref ** 2, axis=1))
    assert np.allclose(-xs @ m.T, ref, rtol=0, atol=1e-9 * np.abs(ref).max())
    assert (np.sqrt(np.mean(((two - xs) @ m.T) ** 2, axis=1)) / size).max() > 1e-6
    h = backend.upload_weight(Q4_K, w, k, rows)
    Y = h.launch_only_batch(torch.from_numpy(X).cuda(), mode=gq.GQ_GEMM_INT8).cpu().numpy()
    check_tokens(Y, ref, 5e-7)


@pytest.mark.parametrize("dtype", [Q4_K, Q6_K])
def test_gemm_int8_scale_overflow(backend, orc, dtype):
    """A block whose f16 scale overflows gives infinite products: results of
    one sign stay infinite, and other tokens finite.  (Q4_K with a negative
    dmin, so that the min term has the dot's sign.)"""
    import gq
    import torch
    rows, k, n = 37, 512, 5
    w = syn.make_blocks(dtype, rows, k, seed=81)
    if dtype == Q4_K:
        b = w.reshape(rows, -1, 144)
        b[..., 0:4] = np.array([0.01, -0.01], np.float16).view(np.uint8)
        b[..., 4:16] = 0x21  # scales and mins 33 or more than 0
    else:
        b = w.reshape(rows, -1, 210)
        b[..., 128:192] |= 0xAA  # codes above 32
        b[..., 0:128] |= 0x11
        b[..., 192:208] = 5
    X = syn.make_x(k, seed=82, batch=n)
    X[1, 64:96] = 1e7
    X[3, 256:288] = -1e7
    h = backend.upload_weight(dtype, w, k, rows)
    Y = h.launch_only_batch(torch.from_numpy(X).cuda(), mode=gq.GQ_GEMM_INT8).cpu().numpy()
    assert np.all(Y[1] == np.inf) and np.all(Y[3] == -np.inf)
    fin = [0, 2, 4]
    check(Y[fin], int8_ref(orc, dtype, w, X[fin]), "other tokens")


@pytest.mark.parametrize("mode,dtype,rows,k,n", [(0, Q4_K, 10611, 256, 959), (0, Q4_K, 40003, 512, 128),
                                                 (1, Q6_K, 10611, 512, 959), (1, Q4_K, 3891, 256, 987)])
def test_gemm_odd_rows(backend, mode, dtype, rows, k, n):
    """Row counts other than 4 m: results start at any dword, at no cost of a
    store per element (10611 x 512 Q6_K at 959 tokens: 81 us with that, 59
    without, 59 for 10612 rows), and the rows past the last are not written."""
    import torch
    say(f"gemm odd rows mode={mode} dtype={dtype} rows={rows} k={k} n={n}")
    w = syn.make_blocks(dtype, rows + 1, k, seed=93)
    X = torch.from_numpy(syn.make_x(k, seed=94, batch=n)).cuda()
    us, got = [], []
    for r in (rows, rows + 1):
        assert r == rows or r % 4 == 0
        h = backend.upload_weight(dtype, np.ascontiguousarray(w[:r]), k, r)
        buf = torch.full((n * r + 9,), 7.0, device="cuda")
        Y = buf[1:1 + n * r].view(n, r)
        t = []
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                h.launch_only_batch(X, mode=mode, Y_dev=Y)
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b) / 20 * 1e3)
        us.append(min(t))
        assert buf[0] == 7.0 and torch.all(buf[1 + n * r:] == 7.0)
        got.append(Y)
    assert torch.equal(got[0], got[1][:, :rows])
    say(f"  {us[0]:.1f} us, {us[1]:.1f} for one row more")
    assert us[0] <= 1.15 * us[1]


def test_gemm_full_config(backend, orc):
    """config 2: Q4_K 18944 x 3584 times 512 tokens, both modes."""
    import gq
    import torch
    rows, k, n = 18944, 3584, 512
    say("gemm full config 18944x3584x512")
    w = syn.make_blocks(Q4_K, rows, k, seed=42)
    X = syn.make_x(k, seed=43, batch=n)
    h = backend.upload_weight(Q4_K, w, k, rows)
    Xd = torch.from_numpy(X).cuda()
    Yb = h.launch_only_batch(Xd, mode=gq.GQ_GEMM_BF16).cpu().numpy()
    Yi = h.launch_only_batch(Xd, mode=gq.GQ_GEMM_INT8).cpu().numpy()
    torch.cuda.synchronize()
    Wf = orc.dequant(Q4_K, w.reshape(-1), rows * k).reshape(rows, k).astype(np.float64)
    ref = bf16_round(X).astype(np.float64) @ bf16_round(Wf.astype(np.float32)).astype(np.float64).T
    check(Yb, ref, "full bf16 vs same-operand fp64")
    Xq = np.zeros((n, k), np.float64)
    for t in range(n):
        sc, q = orc.quantize_q8_32(X[t])
        Xq[t] = q.astype(np.float64) * np.repeat(sc.view(np.float16).astype(np.float64), 32)
    check(Yi, Xq @ Wf.T, "full int8 vs same-operand fp64")
    # the fp32 CPU path (WeightMap::matmul_batch_into) on 16 of the 512
    # tokens: the distance is the operands' rounding (bf16 2^-9 each; per-32
    # Q8 activations 2^-8)
    sub = np.arange(0, n, n // 16)
    ref32 = orc.matmul_batch_into(Q4_K, w, X[sub], rows)
    check(Yb[sub], ref32, "full bf16 vs fp32 CPU path (16 tokens)", tol=1e-2)
    check(Yi[sub], ref32, "full int8 vs fp32 CPU path (16 tokens)", tol=3e-2)


Q8_0, Q5_K = 8, 13
# Q8_0 and Q5_K (bf16 mode only): token counts on both sides of the ring /
# direct kernel boundary (both run the direct kernel), a ragged last unit
# (Q8_0 k = 288), K splits.
OTHER_SHAPES = [(Q8_0, 331, 512, 37), (Q8_0, 1024, 2048, 300), (Q8_0, 100, 288, 20),
                (Q8_0, 8192, 2048, 512), (Q5_K, 331, 512, 37), (Q5_K, 512, 3584, 300),
                (Q5_K, 40, 768, 3)]


@pytest.mark.parametrize("dtype,rows,k,n", OTHER_SHAPES)
def test_gemm_bf16_q8_0_q5k(backend, orc, dtype, rows, k, n):
    """WeightMap::matmul_batch_into (src/model/mod.rs:414-464) dequantizes
    every dtype with dequant_row; the bf16 GEMM of Q8_0 and Q5_K weights
    against the same-operand fp64 product (1e-4) and the fp32 CPU path
    (1e-2, bf16 operands).  (8192 x 2048 is the 1B-class Q8_0 FFN-up
    matrix, here over 512 prompt tokens.)"""
    import gq
    say(f"gemm bf16 dtype={dtype} rows={rows} k={k} n={n}")
    w, X, Wf, Y = run(backend, orc, rows, k, n, gq.GQ_GEMM_BF16, seed=rows + 3 * k + dtype, dtype=dtype)
    ref = bf16_round(X).astype(np.float64) @ bf16_round(Wf).astype(np.float64).T
    check(Y, ref, f"bf16 dtype {dtype} vs same-operand fp64")
    sub = np.arange(0, n, max(1, n // 16))
    ref32 = orc.matmul_batch_into(dtype, w, X[sub], rows)
    check(Y[sub], ref32, f"bf16 dtype {dtype} vs fp32 CPU path", tol=1e-2)


def test_gemm_errors_and_edges(backend):
    import gq
    import torch
    w = syn.make_blocks(13, 4, 256, seed=1)  # Q5_K: bf16 only
    h = backend.upload_weight(13, w, 256, 4)
    with pytest.raises(gq.GqError, match="not supported"):
        h.launch_only_batch(torch.zeros((2, 256), device="cuda"), mode=gq.GQ_GEMM_INT8)
    w8 = syn.make_blocks(8, 4, 256, seed=1)  # Q8_0: bf16 only
    h8 = backend.upload_weight(8, w8, 256, 4)
    with pytest.raises(gq.GqError, match="not supported"):
        h8.launch_only_batch(torch.zeros((2, 256), device="cuda"), mode=gq.GQ_GEMM_INT8)
    w4 = syn.make_blocks(Q4_K, 4, 256, seed=1)
    h4 = backend.upload_weight(Q4_K, w4, 256, 4)
    with pytest.raises(gq.GqError, match="mode"):
        h4.launch_only_batch(torch.zeros((2, 256), device="cuda"), mode=7)
    # n = 0 is a no-op; zero weights give zeros
    h4.launch_only_batch(torch.zeros((0, 256), device="cuda"))
    z = backend.upload_weight(Q4_K, syn.make_blocks(Q4_K, 9, 512, zero=True), 512, 9)
    for mode in (gq.GQ_GEMM_BF16, gq.GQ_GEMM_INT8):
        y = z.launch_only_batch(torch.randn((3, 512), device="cuda"), mode=mode)
        torch.cuda.synchronize()
        assert torch.all(y == 0)



@pytest.mark.parametrize("mode", [0, 1])
def test_gemm_capture_of_shorter_batches(backend, mode):
    """One eager call of the largest batch, in either mode, leaves room for
    capturing any shorter one, also where that splits K further."""
    import torch
    t, rows, k = Q4_K, 18944, 1024
    h = backend.upload_weight(t, syn.make_blocks(t, rows, k, seed=71), k, rows)
    X = torch.from_numpy(syn.make_x(k, seed=72, batch=512)).cuda()
    Y = torch.zeros((512, rows), device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    h.launch_only_batch(X, mode=1 - mode, Y_dev=Y, stream=s.cuda_stream)
    s.synchronize()
    for n in (129, 128, 40):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            h.launch_only_batch(X[:n], mode=mode, Y_dev=Y[:n], stream=s.cuda_stream)
        ref = torch.zeros((n, rows), device="cuda")
        h.launch_only_batch(X[:n], mode=mode, Y_dev=ref, stream=s.cuda_stream)
        s.synchronize()
        for i in range(2):
            Y.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(Y[:n], ref), f"n {n} replay {i}"


def test_gemm_growing_batch_keeps_little(backend):
    """Batches that grow on one stream: the workspaces that later ones
    supersede are kept, so only a few sizes may be taken."""
    import torch
    rows, k = 18944, 3584
    h = backend.upload_weight(Q4_K, syn.make_blocks(Q4_K, rows, k, seed=75), k, rows)
    X = torch.from_numpy(syn.make_x(k, seed=76, batch=512)).cuda()
    Y = torch.zeros((512, rows), device="cuda")
    s = torch.cuda.Stream()
    h.launch_only_batch(X[:1], Y_dev=Y[:1])  # (the weight's records)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    for n in range(1, 513, 7):
        h.launch_only_batch(X[:n], Y_dev=Y[:n], mode=n % 2, stream=s.cuda_stream)
    s.synchronize()
    kept = free - torch.cuda.mem_get_info()[0]
    say(f"kept {kept / 1e6:.1f} MB")
    assert kept <= 200e6


@pytest.mark.parametrize("mode,rows,k,n0,n", [(1, 600, 512, 1, 256), (1, 600, 512, 300, 512), (0, 41000, 256, 1, 512)])
def test_gemm_capture_of_longer_batches(backend, mode, rows, k, n0, n):
    """A warm-up with fewer tokens leaves room for the longer ones that share
    its padding."""
    import torch
    h = backend.upload_weight(Q4_K, syn.make_blocks(Q4_K, rows, k, seed=77), k, rows)
    X = torch.from_numpy(syn.make_x(k, seed=78, batch=n)).cuda()
    Y = torch.zeros((n, rows), device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    h.launch_only_batch(X[:n0], mode=mode, Y_dev=Y[:n0], stream=s.cuda_stream)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        h.launch_only_batch(X, mode=mode, Y_dev=Y, stream=s.cuda_stream)
    ref = h.launch_only_batch(X, mode=mode)
    torch.cuda.synchronize()
    for i in range(2):
        Y.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(Y, ref), f"replay {i}"


def test_gemm_capture_survives_workspace_growth(backend):
    """A HIP graph captured around gq_gemm keeps its workspace: a later,
    larger call on the same stream grows the stream's workspace without
    freeing the captured one, and every replay (with eager work between)
    reproduces the eager result.  Under capture, growing the workspace and
    the first call on a weight (which builds its GEMM records) fail with
    GqError instead of allocating."""
    import torch
    import gq
    rows, k = 1024, 3584
    w = syn.make_blocks(Q4_K, rows, k, seed=61)
    h = backend.upload_weight(Q4_K, w, k, rows)
    h_new = backend.upload_weight(Q4_K, syn.make_blocks(Q4_K, 256, k, seed=64), k, 256)
    s = torch.cuda.Stream()
    Xs = torch.from_numpy(syn.make_x(k, seed=62, batch=64)).cuda()
    Xl = torch.from_numpy(syn.make_x(k, seed=63, batch=512)).cuda()
    Ys = torch.zeros((64, rows), device="cuda")
    Yl = torch.zeros((512, rows), device="cuda")
    Yn = torch.zeros((64, 256), device="cuda")
    torch.cuda.synchronize()
    h.launch_only_batch(Xs, Y_dev=Ys, stream=s.cuda_stream)
    s.synchronize()
    ref = Ys.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        h.launch_only_batch(Xs, Y_dev=Ys, stream=s.cuda_stream)
    for bad, Xb, Yb in ((h, Xl, Yl), (h_new, Xs, Yn)):
        g_bad = torch.cuda.CUDAGraph()
        with pytest.raises(gq.GqError, match="capture"):
            with torch.cuda.graph(g_bad, stream=s):
                bad.launch_only_batch(Xb, Y_dev=Yb, stream=s.cuda_stream)
        torch.cuda.synchronize()
    # the larger call grows the workspace (eager)
    h.launch_only_batch(Xl, Y_dev=Yl, stream=s.cuda_stream)
    s.synchronize()
    ref_l = Yl.clone()
    for i in range(3):
        Ys.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(Ys, ref), f"replay {i}"
        h.launch_only_batch(Xl, Y_dev=Yl, stream=s.cuda_stream)
        s.synchronize()
        assert torch.equal(Yl, ref_l)
