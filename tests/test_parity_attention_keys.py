"""GPU parity: the attention kernel whose waves divide the keys (few queries, or few (head, query tile) pairs), and the merge
of a division of the keys between workgroups, against 64-bit attention of the same 16-bit operands.

Bound of every element: the weights are rounded to the operand type before the second product and the result once after it,
each by at most u (half a unit in the last place, relative), so |error| <= 2 u sum(w |v|); the sums in fp32 and the base-2
weights (some 1e-6) are covered by a tenth more."""
import numpy as np
import pytest

from dvm_amd.tester import Tester
from tests.test_parity_attention import attention_graph

pytestmark = pytest.mark.gpu


def _check(q, k, v, dt, keys, parts, out=None):
    d, scale = q.shape[-1], 1.0 / np.sqrt(q.shape[-1])
    t = Tester("mix")
    dts = dt if dt == "bfloat16" else None
    if dt == "bfloat16":
        q, k, v = (Tester.convert_from_bf16(Tester.convert_to_bf16(x.astype(np.float32))) for x in (q, k, v))
    lq, lk, lv = t.load(q, dts), t.load(k, dts), t.load(v, dts)
    if out == "seq_first":  # operands and result as [batch, tokens, heads, d] in memory
        lq, lk, lv = (t.permute(x, [0, 2, 1, 3]) for x in (lq, lk, lv))
        q, k, v = (x.transpose(0, 2, 1, 3) for x in (q, k, v))
    o = attention_graph(t, lq, lk, lv, scale, q.ndim, dt)
    st = t.store(t.permute(o, [0, 2, 1, 3]) if out == "seq_first" else o)
    t.run()
    if keys is not None:
        assert ("waves divide the keys" in t.das()) == keys, t.das()
    if parts is not None:
        assert t.num_launches() == (2 if parts > 1 else 1) and "parts=%d" % parts in t.das(), t.das()
    got = t.output(st)
    got = (Tester.convert_from_bf16(got) if dt == "bfloat16" else got).astype(np.float64)
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    s = np.matmul(q, np.swapaxes(k, -1, -2)) * scale
    w = np.exp(s - s.max(-1, keepdims=True))
    w /= w.sum(-1, keepdims=True)
    want, bound = np.matmul(w, v), np.matmul(w, np.abs(v))
    if out == "seq_first":
        want, bound = want.transpose(0, 2, 1, 3), bound.transpose(0, 2, 1, 3)
    u = 2.0 ** -9 if dt == "bfloat16" else 2.0 ** -11
    err = np.abs(got - want)
    assert (err <= 2.2 * u * bound + 2.0 ** -24).all(), (err / bound).max()


@pytest.mark.parametrize("dt", ["float16", "bfloat16"])
@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("sq,skv", [(1, 1), (1, 31), (2, 32), (5, 33), (32, 127), (33, 128), (31, 129), (65, 257), (1, 1000)])
def test_attention_keys_edges_of_blocks_and_tiles(monkeypatch, sq, skv, d, dt):
    # every wave with and without a block, a last block of one key and of all, one query and one past a tile
    monkeypatch.setenv("DVM_ATTN_KEYS", "1")
    rng = np.random.default_rng(sq * 10000 + skv + d)
    q, k = (rng.standard_normal((3, n, d)).astype(np.float16) for n in (sq, skv))
    _check(q, k, (rng.standard_normal((3, skv, d)) * 4).astype(np.float16), dt, True, 1)


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("sq,skv,ask,parts", [(1, 129, 2, 2), (3, 1000, 4, 4), (33, 700, 5, 3), (8, 2049, 32, 17), (40, 128, 8, 1)])
def test_attention_keys_in_parts(monkeypatch, sq, skv, ask, parts, d):
    # parts of whole steps (128 keys), the last one down to one key; spread scores, so that the parts' maxima differ
    monkeypatch.setenv("DVM_ATTN_KEYS", str(ask))
    rng = np.random.default_rng(skv + d)
    q, k, v = ((rng.standard_normal((2, n, d)) * m).astype(np.float16) for n, m in ((sq, 4.0), (skv, 1.0), (skv, 4.0)))
    _check(q, k, v, "float16", True, parts)


@pytest.mark.parametrize("b,h,sq,skv,d,dt", [(2, 3, 1, 400, 128, "bfloat16"), (3, 5, 4, 90, 64, "float16"), (1, 4, 300, 300, 128, "float16")])
@pytest.mark.parametrize("ask", ["1", "4"])
def test_attention_keys_on_sequence_major_tensors(monkeypatch, b, h, sq, skv, d, dt, ask):
    monkeypatch.setenv("DVM_ATTN_KEYS", ask)
    rng = np.random.default_rng(b * 100 + h)
    _check(*(rng.standard_normal((b, n, h, d)).astype(np.float16) for n in (sq, skv, skv)), dt, True, None, out="seq_first")


@pytest.mark.parametrize("heads,sq,skv,d,keys,parts", [(4, 1, 4096, 128, True, None), (512, 1, 500, 64, True, 1), (4, 2000, 300, 128, True, 1), (64, 600, 600, 128, False, None)])
def test_attention_keys_rule(heads, sq, skv, d, keys, parts):
    rng = np.random.default_rng(heads)
    _check(*(rng.standard_normal((heads, n, d)).astype(np.float16) for n in (sq, skv, skv)), "float16", keys, parts)


def test_attention_keys_scores_of_minus_infinity_and_nan(monkeypatch):
    # a key whose score is -inf has no weight, also beside masked keys past the end and in a part of its own; a query
    # whose scores hold NaN gives NaN
    rng = np.random.default_rng(5)
    for ask in ("1", "2"):
        monkeypatch.setenv("DVM_ATTN_KEYS", ask)
        q, k, v = (rng.standard_normal((1, n, 64)).astype(np.float16) for n in (2, 161, 161))
        q[0, :, 0] = 1.0
        k[0, 128:, 0] = -np.inf  # the whole second part, and the block that ends in masked keys
        t = Tester("mix")
        st = t.store(attention_graph(t, t.load(q), t.load(k), t.load(v), 0.125, 3))
        t.run()
        s = np.matmul(q[0].astype(np.float64), k[0, :128].T.astype(np.float64)) * 0.125
        w = np.exp(s - s.max(-1, keepdims=True))
        want = np.matmul(w / w.sum(-1, keepdims=True), v[0, :128].astype(np.float64))
        assert np.allclose(t.output(st)[0], want, rtol=0, atol=2.2 * 2.0 ** -11 * np.abs(v.astype(np.float64)).max())
        q[0, 1, 3] = np.nan
        t = Tester("mix")
        st = t.store(attention_graph(t, t.load(q), t.load(k), t.load(v), 0.125, 3))
        t.run()
        got = t.output(st)[0]
        assert np.isnan(got[1]).all() and np.allclose(got[0], want[0], rtol=0, atol=2.2 * 2.0 ** -11 * np.abs(v.astype(np.float64)).max())
