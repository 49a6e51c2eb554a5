"""The few-token projections (gemm_kw.hip: K split over the waves of a block)
through the C ABI against float64, at the edges of their tiles and of the rule
that picks them: every output tile, ragged tokens and rows, K shorter than the
block's waves, prepared matrices and matrices in their own format, groups
longer than a launch, and operands whose alignment the kernels do not take."""
import ctypes

import numpy as np
import pytest

from parity import parity
from qwen_mi355x.bridge import Bridge, pack_bf16, pack_int8

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    b = Bridge()
    yield b
    b.close()


def matrix(kind, w, rows, cols):
    """(the words as uploaded, the values in float64, the row scales)."""
    if kind == "f32":
        return w, w.reshape(rows, cols).astype(np.float64), np.ones(rows)
    if kind == "bf16":
        dense = ((w.view(np.uint32) >> 16) << 16).view(np.float32)
        return pack_bf16(w), dense.reshape(rows, cols).astype(np.float64), np.ones(rows)
    s, q = O.quantize_int8_rows(w, rows, cols)
    return pack_int8(s, q), q.reshape(rows, cols).astype(np.float64), s.astype(np.float64)


def near(got, X, W, scale):
    """fp32 sums: |error| <= 2e-5 sum |x w|, the projections' bound."""
    want = (X @ W.T) * scale[None]
    bound = (np.abs(X) @ np.abs(W).T) * np.abs(scale)[None] * 2e-5 + 1e-30
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) / bound)


# rows x cols at batch: the tile each takes (tokens x rows) or why it is here
SHAPES = [(1024, 3584, 5), (1024, 2048, 128), (1024, 1024, 129),  # 32x16 up to 256 blocks, 32x32 past them
          (2048, 1024, 77), (5120, 1024, 65), (6144, 1024, 128), (1024, 3584, 300),  # 32x64 / 64x32, 64x64
          (6144, 1024, 640), (6144, 1024, 641),  # the rule's last token count and the next
          (33, 32, 31), (7, 96, 33), (130, 160, 64), (16, 1024, 23), (127, 64, 640)]  # ragged rows, few k tiles


@pytest.mark.parametrize("kind", ["f32", "bf16", "i8"])
@pytest.mark.parametrize("prepared", [True, False])
@pytest.mark.parametrize("rows,cols,batch", SHAPES)
def test_projection(gpu, kind, prepared, rows, cols, batch):
    print(f"few tokens {kind} {rows}x{cols} batch {batch} prepared {prepared}", flush=True)
    rng = np.random.default_rng(rows + cols + batch)
    words, W, scale = matrix(kind, (rng.standard_normal(rows * cols) * 0.02).astype(np.float32), rows, cols)
    x = rng.standard_normal(batch * cols).astype(np.float32)
    a, xb, y = gpu.upload(words), gpu.upload(x), gpu.alloc(batch * rows)
    if prepared:
        gpu.prepare(a, rows, cols, kind=kind)
    gpu.gemm(y, a, xb, rows, cols, batch, kind=kind)
    first = y.read()
    near(first.reshape(batch, rows), x.reshape(batch, cols).astype(np.float64), W, scale)
    gpu.gemm(y, a, xb, rows, cols, batch, kind=kind)
    assert np.array_equal(first, y.read())


@pytest.mark.parametrize("kind", ["f32", "bf16", "i8"])
@pytest.mark.parametrize("prepared", [True, False])
@pytest.mark.parametrize("rows,batch", [(3584, 5), (3584, 32), (3584, 77), (3584, 300), (3584, 640), (32, 33), (96, 64)])
def test_glu(gpu, kind, prepared, rows, batch):
    """silu(x G^T) * (x U^T) against the two projections' float64 values, and
    the down projection right after it (over the planes the GLU wrote) equal to
    the one after another call (which splits the product again)."""
    print(f"few tokens glu {kind} {rows} batch {batch} prepared {prepared}", flush=True)
    rng = np.random.default_rng(rows + batch)
    cols, out = 1024, 256
    ws = [(rng.standard_normal(n) * 0.02).astype(np.float32) for n in (rows * cols, rows * cols, out * rows)]
    shapes = [(rows, cols), (rows, cols), (out, rows)]
    mats, values = [], []
    for w, (r, c) in zip(ws, shapes):
        words, W, scale = matrix(kind, w, r, c)
        mats.append(gpu.upload(words))
        values.append(W * scale[:, None])
        if prepared:
            gpu.prepare(mats[-1], r, c, kind=kind)
    x = rng.standard_normal(batch * cols).astype(np.float32)
    xb, prod, gy, uy = gpu.upload(x), gpu.alloc(batch * rows), gpu.alloc(batch * rows), gpu.alloc(batch * rows)
    ys = [gpu.alloc(batch * out) for _ in range(2)]
    gpu.gemm(ys[0], mats[2], prod, out, rows, batch, kind=kind)  # the product's width is known from here on
    gpu.glu(prod, gy, uy, mats[0], mats[1], xb, rows, cols, batch, kind=kind)
    gpu.gemm(ys[0], mats[2], prod, out, rows, batch, kind=kind)
    gpu.sync()
    gpu.gemm(ys[1], mats[2], prod, out, rows, batch, kind=kind)
    assert np.array_equal(ys[0].read(), ys[1].read())
    X = x.reshape(batch, cols).astype(np.float64)
    g, u = X @ values[0].T, X @ values[1].T
    parity(prod.read(), (g / (1 + np.exp(-g)) * u).reshape(-1), where=f"glu {kind} {rows}x{batch}")


@pytest.mark.parametrize("kind", ["f32", "bf16", "i8"])
def test_group_longer_than_a_launch(gpu, kind):
    """Eleven matrices of one input, prepared and not, of 16 to 200 rows."""
    rng = np.random.default_rng(3)
    cols, batch = 256, 37
    rows = [200, 16, 64, 48, 130, 32, 96, 16, 66, 128, 40]
    mats = [matrix(kind, (rng.standard_normal(r * cols) * 0.02).astype(np.float32), r, cols) for r in rows]
    bufs = [gpu.upload(m[0]) for m in mats]
    for i, (b, r) in enumerate(zip(bufs, rows)):
        if i % 3 == 0:
            gpu.prepare(b, r, cols, kind=kind)
    x = rng.standard_normal(batch * cols).astype(np.float32)
    ys = [gpu.alloc(batch * r) for r in rows]
    gpu.group(list(zip(ys, bufs, rows)), gpu.upload(x), cols, batch, kind=kind)
    for y, m, r in zip(ys, mats, rows):
        near(y.read().reshape(batch, r), x.reshape(batch, cols).astype(np.float64), m[1], m[2])


class At:
    """An address inside a buffer."""

    def __init__(self, buf, words):
        self.buf, self.ptr = buf, buf.at(words)


@pytest.mark.parametrize("kind", ["f32", "bf16", "i8"])
def test_operands_off_alignment(gpu, kind):
    """x, the matrix or the output off 16-byte alignment, and an int8 matrix of
    an odd number of rows: the same values by whichever kernel takes them."""
    rng = np.random.default_rng(9)
    rows, cols, batch = 65, 64, 20
    words, W, scale = matrix(kind, (rng.standard_normal(rows * cols) * 0.02).astype(np.float32), rows, cols)
    x = rng.standard_normal(batch * cols).astype(np.float32)
    X = x.reshape(batch, cols).astype(np.float64)
    a = gpu.upload(np.concatenate([np.zeros(1, np.uint32), words.view(np.uint32)]))
    plain, xo = gpu.upload(words), gpu.upload(np.concatenate([np.zeros(1, np.float32), x]))
    xb, y = gpu.upload(x), gpu.alloc(batch * rows + 1)
    for m, v, o in ((plain, At(xo, 1), y), (At(a, 1), xb, y), (plain, xb, At(y, 1)), (plain, xb, y)):
        gpu.gemm(o, m, v, rows, cols, batch, kind=kind)
        got = y.read()[1:] if isinstance(o, At) else y.read(batch * rows)
        near(got.reshape(batch, rows), X, W, scale)


@pytest.mark.parametrize("kind", ["f32", "bf16", "i8"])
@pytest.mark.parametrize("prepared", [True, False])
@pytest.mark.parametrize("rows,cols,batch", [(16, 1024, 5), (16, 1024, 128), (16, 1024, 640), (16, 96, 33), (10, 32, 23),
                                             (1, 160, 64), (7, 1024, 31), (16, 2048, 77)])
def test_few_rows(gpu, kind, prepared, rows, cols, batch):
    """A matrix of at most 16 rows (the DeltaNet a and b): whole fp32 products,
    the same bits alone and beside wider matrices (200 rows: the narrow tiles'
    sizes; 5120: the widest), the wider ones unchanged by its company."""
    print(f"few rows {kind} {rows}x{cols} batch {batch} prepared {prepared}", flush=True)
    rng = np.random.default_rng(rows + cols + batch)
    x = rng.standard_normal(batch * cols).astype(np.float32)
    X, xb = x.reshape(batch, cols).astype(np.float64), gpu.upload(x)
    mats = {r: matrix(kind, (rng.standard_normal(r * cols) * 0.02).astype(np.float32), r, cols)
            for r in (rows, 200, 5120)}
    bufs = {r: gpu.upload(m[0]) for r, m in mats.items()}
    if prepared:
        for r in (200, 5120):
            gpu.prepare(bufs[r], r, cols, kind=kind)
    alone = gpu.alloc(batch * rows)
    gpu.gemm(alone, bufs[rows], xb, rows, cols, batch, kind=kind)
    near(alone.read().reshape(batch, rows), X, *mats[rows][1:])
    for wide in (200, 5120):
        ys = [gpu.alloc(batch * r) for r in (wide, rows, rows)]
        gpu.group([(ys[0], bufs[wide], wide), (ys[1], bufs[rows], rows), (ys[2], bufs[rows], rows)], xb, cols, batch,
                  kind=kind)
        near(ys[0].read().reshape(batch, wide), X, *mats[wide][1:])
        for y in ys[1:]:
            assert np.array_equal(y.read(), alone.read()), wide


@pytest.mark.parametrize("kind", ["f32", "bf16", "i8"])
def test_few_rows_keep_infinities(gpu, kind):
    """Beside wider matrices the few-row ones keep an infinite input infinite
    and the largest fp32 values finite (their BF16 parts are not)."""
    rows, cols, batch = 16, 1024, 40
    rng = np.random.default_rng(5)
    words, W, scale = matrix(kind, (0.01 + rng.random(rows * cols) * 0.02).astype(np.float32), rows, cols)
    wide = matrix(kind, (rng.standard_normal(512 * cols) * 0.02).astype(np.float32), 512, cols)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    x[3, 700] = np.inf
    x[17, 5] = -np.inf
    x[33, 9] = np.finfo(np.float32).max
    if kind == "i8":
        x[33, 9] /= 256  # (the integers' products are scaled after the sum)
    ys = [gpu.alloc(batch * r) for r in (512, rows)]
    gpu.group([(ys[0], gpu.upload(wide[0]), 512), (ys[1], gpu.upload(words), rows)], gpu.upload(x.reshape(-1)), cols,
              batch, kind=kind)
    got = ys[1].read().reshape(batch, rows)
    assert np.all(got[3] == np.inf) and np.all(got[17] == -np.inf)
    rest = [t for t in range(batch) if t not in (3, 17)]
    near(got[rest], x[rest].astype(np.float64), W, scale)


@pytest.mark.parametrize("batch", [23, 128])
def test_unprepared_inputs_may_be_rewritten(gpu, batch):
    """Where no matrix is prepared, a projection takes its input as it lies in
    memory: also what another context wrote there after the norm or the GLU
    that produced it, with no call of this context in between."""
    cols, rows = 1024, 256
    rng = np.random.default_rng(batch)
    b = Bridge()
    other = Bridge()
    try:
        words, W, scale = matrix("i8", (rng.standard_normal(rows * cols) * 0.02).astype(np.float32), rows, cols)
        square, _, _ = matrix("i8", (rng.standard_normal(cols * cols) * 0.02).astype(np.float32), cols, cols)
        a, sq = b.upload(words), b.upload(square)
        x, norm = b.upload(rng.standard_normal(batch * cols).astype(np.float32)), b.upload(np.zeros(cols, np.float32))
        normed, gy, uy, y = b.alloc(batch * cols), b.alloc(batch * cols), b.alloc(batch * cols), b.alloc(batch * rows)
        producers = [lambda: b.run("RMS_NORM", batch, [normed, x, norm], [cols], [1e-6, 1.0]),
                     lambda: b.glu(normed, gy, uy, sq, sq, x, cols, cols, batch, kind="i8")]
        for produce in producers:
            for _ in range(2):
                produce()
                b.gemm(y, a, normed, rows, cols, batch, kind="i8")
            new = rng.standard_normal(batch * cols).astype(np.float32)
            produce()
            assert b.L.hipDeviceSynchronize() == 0
            assert other.L.qr_write(other.ctx, ctypes.c_void_p(normed.ptr), new.ctypes.data_as(ctypes.c_void_p),
                                    ctypes.c_size_t(new.size)) == 0
            b.gemm(y, a, normed, rows, cols, batch, kind="i8")
            near(y.read().reshape(batch, rows), new.reshape(batch, cols).astype(np.float64), W, scale)
    finally:
        b.close()
        other.close()


@pytest.mark.parametrize("kind", ["f32", "bf16", "i8"])
@pytest.mark.parametrize("rows,cols,bound", [(512, 1024, 1.1e-7), (5120, 1024, 1.1e-7), (1024, 3584, 1.5e-7)])
def test_sums_round_once_per_step(gpu, kind, rows, cols, bound):
    """The error of a projection of a few tokens (2-norm, against float64). A
    rounding of fp32 is about 2.4e-8 of the value (2-norm); n additions to a sum
    that grows as a random walk make 2.4e-8 sqrt(n / 2): 7e-8 for the 16 leading
    products of a wave at K = 1024, 9e-8 for the 28 of a chain at K = 3584, and
    half as much again within the MFMAs (measured 9.8e-8 and 1.28e-7 at most).
    With every part product in the same sums n is three to six times as large
    (fp32: 1.7e-7 and 3.2e-7)."""
    rng = np.random.default_rng(rows + cols)
    e2 = w2 = 0.0
    for batch in (8, 20):
        words, W, scale = matrix(kind, (rng.standard_normal(rows * cols) * 0.02).astype(np.float32), rows, cols)
        x = rng.standard_normal(batch * cols).astype(np.float32)
        y = gpu.alloc(batch * rows)
        gpu.gemm(y, gpu.upload(words), gpu.upload(x), rows, cols, batch, kind=kind)
        want = (x.reshape(batch, cols).astype(np.float64) @ W.T) * scale[None]
        e2 += np.sum((y.read().reshape(batch, rows) - want) ** 2)
        w2 += np.sum(want ** 2)
    print(f"error {np.sqrt(e2 / w2):.3e}", flush=True)
    assert np.sqrt(e2 / w2) < bound
