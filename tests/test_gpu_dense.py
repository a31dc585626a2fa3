"""Dense F32 / F16 / BF16 batches above 8 on the matrix-core GEMM
(nya_hip_matmul, kernel "dense_gemm"), through the kernel library's C ABI:

- under the reference kernel contract (backend/tests/test_quant_kernels.c:13-25,
  :138-213): every token and row within 1e-6 (1 + sum |w x|) of the double
  sum of the decoded products, and within relative L2 1e-5 of the scalar
  oracle (the reference's F32 path accumulates in double,
  backend/core/llm_quant.c:161-204), at batches 9 .. 512, rows that are not
  a multiple of the 128-row tile, tokens that are not a multiple of 64, and
  column counts with a short last 32-column chunk or rows that are not
  16-byte aligned (the element-by-element loads);
- an exact fixture: small integer weights and activations, whose products
  and sums are exact in fp32, give the exact integer result;
- canaries on both sides of the output stay untouched;
each with the workspace nya_hip_workspace_bytes asks for (small tile counts
split the columns over several workgroups, added in order by a second
launch) and without one (a workgroup per tile over all columns).
"""
import numpy as np
import pytest

from fyodor_amd import BF16, F16, F32, TYPE_NAMES, storage_bytes, synth
from fyodor_amd.hip import Kernels, Runtime
from oracle import host_threads

pytestmark = pytest.mark.gpu

SHAPES = [(300, 1024, 9), (129, 1000, 40), (1000, 8192, 65), (64, 33, 17), (100, 1002, 12), (4096, 4096, 512),
          (257, 4104, 100)]


@pytest.fixture(scope="module")
def hip():
    rt = Runtime()
    return rt, Kernels(), rt.stream()


def run(hip, w, t, x, rows, cols, batch, workspace=True):
    """nya_hip_matmul on device copies; the output with one canary float on
    each side. With the workspace it asks for, small tile counts split the
    columns over several workgroups; without, one workgroup per tile."""
    rt, kern, stream = hip
    assert kern.kernel_name(t, rows, cols, batch) == "dense_gemm"
    need = kern.workspace_bytes(t, rows, cols, batch) if workspace else 0
    wd, xd = rt.malloc(max(w.nbytes, 16)), rt.malloc(x.nbytes)
    out, ws = rt.malloc(4 * (batch * rows + 2)), rt.malloc(max(need, 16))
    try:
        rt.upload(wd, w)
        rt.upload(xd, np.ascontiguousarray(x, dtype=np.float32))
        rt.upload(out, np.full(batch * rows + 2, 12345.0, dtype=np.float32))
        kern.matmul(wd, t, rows, cols, xd, out + 4, batch, ws if need else 0, need, stream)
        rt.sync(stream)
        y = rt.download(out, np.empty(batch * rows + 2, dtype=np.float32))
    finally:
        for p in (wd, xd, out, ws):
            rt.free(p)
    assert y[0] == 12345.0 and y[-1] == 12345.0, "canary overwritten"
    return y[1:-1].reshape(batch, rows)


@pytest.mark.parametrize("t", [F32, F16, BF16], ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("rows,cols,batch", SHAPES, ids=[f"{r}x{c}-m{b}" for r, c, b in SHAPES])
def test_dense_gemm_contract(hip, oracle, t, rows, cols, batch):
    seed = 41 * t + rows + cols + batch
    w = synth.weights(t, rows, cols, seed)
    x = synth.activations(batch, cols, seed + 1)
    s, m = oracle.contract_sums(w, t, x, rows, cols)
    scalar = oracle.matmul(w, t, x, rows, cols, batch, threads=host_threads())
    for workspace in (True, False):
        print(f"dense_gemm {TYPE_NAMES[t]} {rows}x{cols} batch {batch} workspace {workspace}", flush=True)
        y = run(hip, w, t, x, rows, cols, batch, workspace)
        assert np.all(np.isfinite(y))
        err = np.abs(y.astype(np.float64) - s)
        bad = err > 1e-6 * (1 + m)
        assert not bad.any(), f"{int(bad.sum())} outputs outside the contract bound, first at {np.argwhere(bad)[0]}"
        num = np.linalg.norm(y.astype(np.float64) - scalar, axis=1)
        den = np.linalg.norm(scalar.astype(np.float64), axis=1)
        assert np.all(num <= 1e-5 * den), f"relative L2 {float((num / den).max()):.3g}"


@pytest.mark.parametrize("t", [F32, F16, BF16], ids=lambda t: TYPE_NAMES[t])
def test_dense_gemm_exact_integers(hip, t):
    """Weights in -8..7 and activations in -16..15: every product and every
    partial sum is an integer below 2^24, so fp32 accumulation is exact."""
    rows, cols, batch = 200, 2048, 70
    rng = np.random.default_rng(7 + t)
    wv = rng.integers(-8, 8, size=(rows, cols)).astype(np.float32)
    x = rng.integers(-16, 16, size=(batch, cols)).astype(np.float32)
    if t == F32:
        w = wv.view(np.uint8).reshape(-1).copy()
    elif t == F16:
        w = wv.astype(np.float16).view(np.uint8).reshape(-1).copy()
    else:
        w = (wv.view(np.uint32) >> 16).astype(np.uint16).view(np.uint8).reshape(-1).copy()
    assert w.nbytes == storage_bytes(t, rows, cols)
    exact = x.astype(np.float64) @ wv.astype(np.float64).T
    for workspace in (True, False):
        y = run(hip, w, t, x, rows, cols, batch, workspace)
        assert np.array_equal(y.astype(np.float64), exact)


def stored(t, v):
    """fp32 values as stored type t (bytes) and the values it holds."""
    if t == F32:
        return v.view(np.uint8).reshape(-1).copy(), v
    if t == F16:
        h = v.astype(np.float16)
        return h.view(np.uint8).reshape(-1).copy(), h.astype(np.float32)
    h = (v.view(np.uint32) >> 16).astype(np.uint16)
    return h.view(np.uint8).reshape(-1).copy(), (h.astype(np.uint32) << 16).view(np.float32)


# Columns about the 64-column step, its halves between the two column groups
# (an odd number of steps, one step, a step of one column) and unaligned rows;
# tokens and rows about their tiles of 64 and 128.
EDGES = [(127, 8, 9), (128, 63, 64), (1, 64, 65), (129, 65, 63), (130, 136, 9), (257, 192, 130), (5, 321, 66), (131, 330, 65),
         (128, 1096, 64), (128, 2184, 10),
         # Short rows on the fp32 cores: their 32-column chunks, the longest that
         # take them in one and in several workgroups per CU, and the next ones.
         (70, 31, 66), (129, 32, 70), (65, 33, 65), (127, 96, 100), (130, 160, 64), (130, 161, 64), (66, 168, 65),
         (140, 320, 40), (140, 324, 40), (4100, 192, 520), (4100, 200, 520), (2100, 448, 1000)]


@pytest.mark.parametrize("t", [F32, F16, BF16], ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("wscale,xscale", [(0, 0), (-14, 90), (-112, 100), (100, -122)])
def test_dense_gemm_pieces(hip, t, wscale, xscale):
    """Values across the exponent range, weights and activations that take
    every bit of their pieces. Products left out weigh below 2^-25 of their
    own magnitude, and a sum of n / 16 partial results rounds at most that
    often: (n / 16 + 16) 2^-24 of sum |w x|."""
    if t == F16:
        wscale = max(wscale, -14) if wscale < 0 else min(wscale, 12)
    for rows, cols, batch in EDGES:
        rng = np.random.default_rng(rows + cols + batch + t)
        wv = np.ldexp(rng.uniform(-1, 1, (rows, cols)) * 2.0 ** rng.integers(-8, 1, (rows, cols)), wscale).astype(np.float32)
        x = np.ldexp(rng.uniform(-1, 1, (batch, cols)) * 2.0 ** rng.integers(-8, 1, (batch, cols)), xscale).astype(np.float32)
        w, wv = stored(t, wv)
        exact = x.astype(np.float64) @ wv.astype(np.float64).T
        bound = (cols / 16 + 16) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(wv).astype(np.float64).T)
        for workspace in (True, False):
            y = run(hip, w, t, x, rows, cols, batch, workspace)
            bad = np.abs(y - exact) > bound
            assert not bad.any(), (rows, cols, batch, workspace, int(bad.sum()))


@pytest.mark.parametrize("t", [F32, F16, BF16], ids=lambda t: TYPE_NAMES[t])
def test_dense_gemm_non_finite(hip, t):
    """Infinities, NaN and the largest values give what a plain sum gives:
    the same infinities and NaN in the same outputs, the others untouched."""
    rows, cols, batch = 130, 200, 70
    rng = np.random.default_rng(t + 1)
    wv = rng.uniform(-1, 1, (rows, cols)).astype(np.float32)
    x = rng.uniform(-1, 1, (batch, cols)).astype(np.float32)
    wv[3, 199], wv[64, 0], wv[129, 100], wv[7, 50], wv[7, 51] = np.inf, -np.inf, np.nan, np.inf, np.inf
    x[0, 64], x[9, 199], x[63, 5], x[69, 150] = np.inf, 0.0, -np.inf, np.nan
    x[20], x[30], x[40:48] = 0.0, 1e-40, 0.0
    wv[32], wv[60:63], wv[128] = 0.0, 0.0, 0.0
    x[20, 3], x[21, 4] = np.float32(3.4028235e38), np.float32(-3.4e38)
    w, wv = stored(t, wv)
    with np.errstate(invalid="ignore"):
        exact = np.stack([[np.sum(x[b].astype(np.float64) * wv[r].astype(np.float64)) for r in range(rows)]
                          for b in range(batch)])
        m = np.stack([np.sum(np.abs(x[b].astype(np.float64) * wv.astype(np.float64)), axis=1) for b in range(batch)])
    for workspace in (True, False):
        y = run(hip, w, t, x, rows, cols, batch, workspace).astype(np.float64)
        assert np.array_equal(np.isnan(y), np.isnan(exact))
        finite = np.isfinite(exact)
        assert np.array_equal(y[~finite & ~np.isnan(exact)], exact[~finite & ~np.isnan(exact)])
        assert np.all(np.abs(y[finite] - exact[finite]) <= (cols / 16 + 16) * 2.0 ** -24 * m[finite])


@pytest.mark.parametrize("t", [F32, F16, BF16], ids=lambda t: TYPE_NAMES[t])
@pytest.mark.parametrize("kind", ["nan-tokens", "nan-rows", "inf-token", "inf-tokens", "inf-rows", "huge", "masked", "padded",
                                  "tiny", "tiny-rows"])
def test_dense_gemm_reviewed_tiles(hip, t, kind):
    """Inputs of which a tile has more outputs to look at again than are
    computed one by one: whether they stand is told from their tokens' and
    rows' ranges, the rest come one by one or with their whole tile on the fp32
    cores. Infinities and NaN as plain sums give them, the other outputs to the
    bound of test_dense_gemm_pieces."""
    for rows, cols, batch in [(200, 704, 130), (130, 901, 65)]:
        rng = np.random.default_rng(rows + cols + t)
        wv = rng.uniform(-1, 1, (rows, cols)).astype(np.float32)
        x = rng.uniform(-1, 1, (batch, cols)).astype(np.float32)
        if kind == "nan-tokens":
            x[rng.random(batch) < 0.5, 7] = np.nan
        elif kind == "nan-rows":
            wv[rng.random(rows) < 0.5, 9] = np.nan
        elif kind == "inf-token":
            x[40, [3, 650]] = np.inf, 1.0
        elif kind == "inf-tokens":
            x[rng.random(batch) < 0.6, 11], x[::9, 12] = np.inf, -np.inf
        elif kind == "inf-rows":
            wv[rng.random(rows) < 0.3, 600], x[5::7, 600] = -np.inf, 0.0
        elif kind == "huge":
            x[3::16] *= np.float32(2.0 ** 120)
            x[50, 100] = np.float32(3.4028e38)
            wv[:, 100] = np.abs(wv[:, 100]) * np.float32(0.125)
        elif kind == "masked":
            x[rng.random(batch) < 0.5, :400] = 0.0
            wv[rng.random(rows) < 0.7, 400:] = 0.0
            x[::5] = np.where(rng.random((len(x[::5]), cols)) < 0.98, 0.0, x[::5])
        elif kind == "padded":
            x[50:], wv[120:] = 0.0, 0.0
        elif kind == "tiny":
            x[1::2] *= np.float32(2.0 ** -118)
            x[::11, 400:] = np.float32(2.0 ** -130)
        else:
            wv[1::3] *= np.float32(2.0 ** (-14 if t == F16 else -110))
            x[::3] *= np.float32(2.0 ** -20)
            wv[::4, 300:] = 0.0
        w, wv = stored(t, wv)
        with np.errstate(invalid="ignore", over="ignore"):
            exact = np.stack([np.sum(wv.astype(np.float64) * x[b].astype(np.float64), axis=1) for b in range(batch)])
            m = np.stack([np.sum(np.abs(wv.astype(np.float64) * x[b].astype(np.float64)), axis=1) for b in range(batch)])
        finite = np.isfinite(exact) & (np.abs(exact) < 2.0 ** 127)
        for workspace in (True, False):
            print(f"{TYPE_NAMES[t]} {kind} {rows}x{cols} batch {batch} workspace {workspace}", flush=True)
            y = run(hip, w, t, x, rows, cols, batch, workspace).astype(np.float64)
            assert np.array_equal(np.isnan(y), np.isnan(exact))
            assert np.array_equal(y[np.isinf(exact)], exact[np.isinf(exact)])
            assert np.all(y[m == 0] == 0)
            # (2^-149: an output's own last place.)
            assert np.all(np.abs(y[finite] - exact[finite]) <= (cols / 16 + 16) * 2.0 ** -24 * m[finite] + 2.0 ** -149)
