"""One decode row of AttentionRead (op 10) at the edges of its chunks, spans and
merges, for every head dim and group size of the decode kernels, and a prefill
chunk's KV shares, against the CPU op."""
import numpy as np
import pytest

from bridges import rnd
from conftest import ROOT
from parity import parity
from qwen_mi355x.bridge import Bridge

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def both():
    g, c = Bridge(), Bridge(ROOT / "oracle" / "lib" / "libqwen_ops_bridge.so", kind=0)
    yield g, c
    g.close()
    c.close()


def read(br, d, heads, kv, length, rows, data):
    q, k, v, gate = (br.upload(x) for x in data)
    out = br.alloc(rows * heads * d)
    scores = br.alloc(heads * max(length + rows, 16 * (d + 2)))
    br.run("ATTENTION_READ", heads, [out, q, k, v, gate, scores],
           [d, heads, kv, length, length + rows, rows, scores.n // heads])
    return out.read()


@pytest.mark.parametrize("d,heads,kv", [(256, 8, 2), (256, 8, 1), (256, 2, 1), (256, 2, 2), (128, 8, 2), (128, 3, 3),
                                        (128, 8, 1), (64, 4, 2), (64, 8, 1), (64, 4, 1), (32, 4, 1), (16, 4, 2)])
@pytest.mark.parametrize("length", [1, 15, 32, 33, 65, 512, 2049, 4111])
def test_decode_row(both, d, heads, kv, length):
    print(f"decode row d={d} heads={heads}/{kv} length={length}", flush=True)
    rng = np.random.default_rng(d + heads + length)
    data = [rnd(rng, heads * d), rnd(rng, length * kv * d), rnd(rng, length * kv * d), rnd(rng, heads * d)]
    got, want = (read(b, d, heads, kv, length, 1, data) for b in both)
    parity(got, want, where=f"decode row {d} {heads}/{kv} {length}")


@pytest.mark.parametrize("length,rows", [(1, 9), (1, 33), (30, 40), (500, 32), (513, 17), (1000, 65),
                                         (1, 700), (40, 1037)])  # several blocks per CU
def test_shares(both, length, rows):
    """KV shares from one tile each up to the most, rows past a 32-row tile."""
    print(f"shares length={length} rows={rows}", flush=True)
    d, heads, kv = 256, 8, 2
    rng = np.random.default_rng(length + rows)
    n = length + rows
    data = [rnd(rng, rows * heads * d), rnd(rng, n * kv * d), rnd(rng, n * kv * d), rnd(rng, rows * heads * d)]
    got, want = (read(b, d, heads, kv, length, rows, data) for b in both)
    parity(got, want, where=f"shares {length} {rows}")


def test_large_scores(both):
    """Scores of hundreds (one position takes all the weight) and equal scores."""
    d, heads, kv, length = 256, 8, 2, 300
    rng = np.random.default_rng(0)
    for scale in (30.0, 0.0):
        data = [rnd(rng, heads * d) * np.float32(scale), rnd(rng, length * kv * d), rnd(rng, length * kv * d),
                rnd(rng, heads * d)]
        got, want = (read(b, d, heads, kv, length, 1, data) for b in both)
        parity(got, want, where=f"scale {scale}")


@pytest.mark.parametrize("heads,kv,length,rows", [(8, 2, 33, 1), (8, 2, 17, 1), (8, 1, 1, 9), (8, 1, 33, 9)])
def test_infinite_values(both, heads, kv, length, rows):
    """An infinite value at a span's first position reaches its own dim of the
    context and no other, also where the span ends inside a chunk."""
    d = 256
    rng = np.random.default_rng(length + rows)
    n = length + rows
    values = rnd(rng, n * kv * d).reshape(n, kv, d)
    at = (length - 1) // 16 * 16 if rows == 1 else 0
    values[at, :, 3] = np.inf
    values[at, :, 250] = -np.inf
    data = [rnd(rng, rows * heads * d), rnd(rng, n * kv * d), values.reshape(-1), rnd(rng, rows * heads * d)]
    got, want = (read(b, d, heads, kv, length, rows, data).reshape(rows, heads, d) for b in both)
    assert np.all(got[..., 3] == np.inf) and np.all(got[..., 250] == -np.inf)
    rest = [i for i in range(d) if i not in (3, 250)]
    parity(got[..., rest], want[..., rest], where=f"inf {length} {rows}")


@pytest.mark.parametrize("heads,kv,rows", [(8, 1, 12), (16, 2, 9)])
def test_long_rows_sum_in_chunks(both, heads, kv, rows):
    """Equal scores (q = 0) over 1920 positions of values in (0, 1): the context
    is the values' mean, its error that of the sum alone. One chain of 480
    additions per wave is off by about 2^-24 sqrt(480) / 3 / 2 = 2.2e-7 (2-norm;
    partial sums grow evenly, four waves' errors average; measured 1.5e-7), chunks
    of 8 with 60 additions between them by 8e-8 (6.5e-8), the division's 3e-8 included."""
    d, length = 256, 1920
    rng = np.random.default_rng(7)
    n = length + rows
    values = rng.random((n, kv, d)).astype(np.float32)
    data = [np.zeros(rows * heads * d, np.float32), rnd(rng, n * kv * d), values.reshape(-1),
            np.full(rows * heads * d, 40.0, np.float32)]  # sigmoid(40) rounds to 1
    got = read(both[0], d, heads, kv, length, rows, data).reshape(rows, kv, heads // kv, d).astype(np.float64)
    want = np.stack([values[:length + r].astype(np.float64).mean(0) for r in range(rows)])[:, :, None]
    err = np.sqrt(np.sum((got - want) ** 2) / np.sum(np.broadcast_to(want, got.shape) ** 2))
    print(f"error {err:.3e}", flush=True)
    assert err < 1.1e-7, err


@pytest.mark.parametrize("d,heads,kv", [(256, 8, 2), (256, 8, 1), (128, 3, 3), (64, 4, 2)])
@pytest.mark.parametrize("length,dead", [(300, 200), (300, 31), (64, 40), (4111, 4100)])
def test_scores_of_minus_infinity(both, d, heads, kv, length, dead):
    """The first `dead` positions score -inf (whole chunks, spans and merge
    inputs among them): they weigh nothing. All of them: NaN, as the CPU op."""
    rng = np.random.default_rng(d + length + dead)
    q = rnd(rng, heads * d).reshape(heads, d)
    q[:, 0] = np.abs(q[:, 0]) + 0.1
    keys = rnd(rng, length * kv * d).reshape(length, kv, d)
    keys[:dead, :, 0] = -np.inf
    data = [q.reshape(-1), keys.reshape(-1), rnd(rng, length * kv * d), rnd(rng, heads * d)]
    got, want = (read(b, d, heads, kv, length, 1, data) for b in both)
    parity(got, want, where=f"-inf {d} {length} {dead}")
    keys[:, :, 0] = -np.inf
    data[1] = keys.reshape(-1)
    for b in both:
        assert np.isnan(read(b, d, heads, kv, length, 1, data)).all()


@pytest.mark.parametrize("length,rows", [(1, 9), (77, 40), (500, 33)])
def test_rows_of_eight_heads(both, length, rows):
    """Head dim 256 with eight query heads per KV head has no tiled prefill
    form: each row of a chunk is one block over its whole length."""
    print(f"rows of 8 heads length={length} rows={rows}", flush=True)
    d, heads, kv = 256, 8, 1
    rng = np.random.default_rng(length + rows)
    n = length + rows
    data = [rnd(rng, rows * heads * d), rnd(rng, n * kv * d), rnd(rng, n * kv * d), rnd(rng, rows * heads * d)]
    got, want = (read(b, d, heads, kv, length, rows, data) for b in both)
    parity(got, want, where=f"eight heads {length} {rows}")


@pytest.mark.parametrize("length", [2000, 4000])
def test_merge_adds_in_pairs(both, length):
    """Equal scores over 125 splits of values in (0, 1): 16 waves' sums of even
    size. Added in one chain they are off by 2.4e-8 sqrt(16 / 3) = 5.5e-8 (2.4e-8:
    one rounding, 2-norm), in pairs by 2.4e-8 sqrt(1 + 1/2 + 1/4 + 1/8) = 3.3e-8;
    the sums before and the division add 3e-8 (root of squares)."""
    d, heads, kv = 256, 8, 2
    rng = np.random.default_rng(length)
    err = []
    for _ in range(4):
        values = rng.random((length, kv, d)).astype(np.float32)
        data = [np.zeros(heads * d, np.float32), rnd(rng, length * kv * d), values.reshape(-1),
                np.full(heads * d, 40.0, np.float32)]  # sigmoid(40) rounds to 1
        got = read(both[0], d, heads, kv, length, 1, data).reshape(kv, heads // kv, d).astype(np.float64)
        want = np.broadcast_to(values.astype(np.float64).mean(0)[:, None], got.shape)
        err.append(np.sum((got - want) ** 2) / np.sum(want ** 2))
    err = np.sqrt(np.mean(err))
    print(f"error {err:.3e}", flush=True)
    assert err < 5.3e-8


@pytest.mark.parametrize("length,rows,bound", [(1, 128, 1.5e-7), (2001, 1000, 3.6e-7)])
def test_prefill_read_error(both, length, rows, bound):
    """The error of a chunk's read (2-norm, against float64). A score over 256
    dims is two sums of 48 MFMAs; one rounding is about 2.4e-8 of the sum (2-norm)
    and a sum grows as a random walk, so 48 at its size make 2.4e-8 sqrt(48 / 2) =
    1.2e-7 of a score, the 8 leading products alone, after the others, 5e-8.
    Measured here 1.95e-7 and 3.93e-7 with a step's six products together, 1.19e-7
    and 3.19e-7 so; the contexts' own sums are the rest."""
    d, heads, kv = 256, 8, 2
    rng = np.random.default_rng(rows)
    n = length + rows - 1
    data = [rnd(rng, rows * heads * d), rnd(rng, n * kv * d), rnd(rng, n * kv * d), rnd(rng, rows * heads * d)]
    got = read(both[0], d, heads, kv, length, rows, data).reshape(rows, heads, d)
    q, k, v, gate = (x.astype(np.float64) for x in data)
    q, k, v, gate = q.reshape(rows, heads, d), k.reshape(n, kv, d), v.reshape(n, kv, d), gate.reshape(rows, heads, d)
    seen = np.arange(n)[None] < length + np.arange(rows)[:, None]
    e2 = w2 = 0.0
    for h in range(heads):
        s = np.where(seen, q[:, h] @ k[:, h // 4].T / np.sqrt(d), -np.inf)
        s = np.exp(s - s.max(1, keepdims=True))
        want = (s / s.sum(1, keepdims=True)) @ v[:, h // 4] / (1 + np.exp(-gate[:, h]))
        e2 += np.sum((got[:, h] - want) ** 2)
        w2 += np.sum(want ** 2)
    print(f"error {np.sqrt(e2 / w2):.3e}", flush=True)
    assert np.sqrt(e2 / w2) < bound
