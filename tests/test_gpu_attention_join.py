"""Rows of several 2048-position chunks against the softmax over the whole row in float64 (attention_tables), in passes of
one token (lane chains), 16 and 64 tokens (matrix cores)."""
import numpy as np
import pytest

from attention_tables import IDS, Tables

pytestmark = pytest.mark.gpu

ORDINARY = IDS - 8  # ids below it have the tables' random rows; those from it on are set by the tests


def rows_of(m, ids, first, n):
    """Logits of positions `first`.. in passes of n tokens."""
    m.truncate(0)
    for i in range(0, first, 64):
        m.forward_batch(ids[i:min(i + 64, first)], logits="none")
    return np.concatenate([m.forward_batch(ids[i:i + n], logits="all").copy() for i in range(first, len(ids), n)])


def special(case, t, ids):
    """Sets the tables' special ids and places them; the rows whose outputs must not be finite."""
    a, b = ORDINARY, ORDINARY + 1
    t.k[:ORDINARY, -2:] = 0.25
    t.q[:, :, -2:] = 1.0
    if case == "a chunk of NaN":
        # the last key overflows the f16 cache in two dimensions of opposite signs: inf - inf, alone in its chunk
        t.k[a, -2:] = 1e5, -1e5
        ids[2048] = a
    elif case == "first chunk -inf":
        t.k[a, -1] = -1e5
        ids[:2048] = a
    elif case == "middle chunk -inf":
        t.k[a, -1] = -1e5
        ids[2048:4096] = a
    elif case == "every chunk -inf":
        t.k[a, -1] = -1e5
        ids[:] = a
    elif case == "inf at weight 0":
        # one value overflows in a chunk whose scores lie 1000 below the others': 0 times inf
        t.q[:, :, -1] = 100.0
        t.k[:ORDINARY, -1] = 0.0
        t.k[a], t.k[b] = t.k[0], t.k[1]
        t.k[[a, b], -1] = -10.0 * np.sqrt(t.hd)
        t.v[b, 3] = 1e5
        ids[:2048] = a
        ids[1000] = b


@pytest.mark.parametrize("head_dim,kv", [(64, "f16"), (128, "f16"), (256, "f16"), (128, "f32")])
def test_chunks_of_uneven_weight_join_to_the_softmax_of_the_row(gpu, monkeypatch, tmp_path, head_dim, kv):
    """Three chunks whose scores differ by a few units, the last one of about 1000 positions, each with a share of the sum
    that counts: the outputs against float64, and an answer with one chunk lost or given a neighbour's weight is far off."""
    t = Tables(head_dim, 12)
    third = IDS // 3
    t.q[:, :, -1] = 1.0
    for c, score in enumerate((0.0, 1.5, -0.75)):  # of the ids of chunk c
        t.k[c * third:(c + 1) * third, -1] = np.float16(score * np.sqrt(head_dim))
    rng = np.random.default_rng(13)
    ids = np.concatenate([rng.integers(c * third, (c + 1) * third, n) for c, n in enumerate((2048, 2048, 1016))])
    first = len(ids) - 16
    want = t.exact(ids, range(first, len(ids)))
    # float32 scores of at most 8 in all (2^-22 absolute), probabilities rounded twice, and the chain's one rounding of the
    # running sum a position, which add up like sqrt(2048) 2^-24 of sum p |v| (0.8 of a value's standard deviation)
    bound = 2.0 ** -22 + 2.0 ** -23 + 4 * np.sqrt(2048) * 2.0 ** -24
    for lost in range(3):
        keep = np.r_[:lost * 2048, min((lost + 1) * 2048, len(ids)):len(ids)]
        if lost < 2:
            assert np.abs(t.exact(ids[keep], range(len(keep) - 16, len(keep))) - want).max() > 100 * bound
    m = t.load(monkeypatch, str(tmp_path / "t.gguf"), ctx=len(ids) + 8, kv=kv)
    for n in (1, 5, 16):
        print(f"case uneven chunks head {head_dim} kv {kv} passes of {n}", flush=True)
        err = np.abs(t.outputs(rows_of(m, ids.tolist(), first, n), ids[first:]) - want).max()
        print(f"largest error {err:.2e}, bound {bound:.2e}", flush=True)
        assert err <= bound, n
    m.close()


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("case,length", [("a chunk of NaN", 2049), ("a chunk of NaN", 2064), ("first chunk -inf", 2700),
                                         ("middle chunk -inf", 4200), ("every chunk -inf", 2060), ("inf at weight 0", 2700)])
def test_infinities_and_nan_are_those_of_the_whole_row(gpu, monkeypatch, tmp_path, case, length, head_dim):
    t = Tables(head_dim, 3)
    ids = np.random.default_rng(4).integers(0, ORDINARY, length)
    special(case, t, ids)
    first = max(length - 16, 2048)
    m = t.load(monkeypatch, str(tmp_path / "t.gguf"), ctx=length + 3, kv="f16")
    want = t.exact(ids, range(first, length))
    for n in (1, 16, 64):
        print(f"case {case} head {head_dim} passes of {n}", flush=True)
        got = rows_of(m, ids.tolist(), first, n)
        bad = ~np.isfinite(want).all(1)
        assert bad.all() == (case in ("a chunk of NaN", "every chunk -inf", "inf at weight 0")) and bad.all() == bad.any()
        assert (np.isfinite(got).all(1) == ~bad).all(), n
        if not bad.any():
            assert np.abs(t.outputs(got, ids[first:]) - want).max() <= 1e-5 * np.abs(want).max()
    m.close()


@pytest.mark.parametrize("kv", ["f16", "f32"])
@pytest.mark.parametrize("ctx,at", [(1024, 300), (4224, 300), (4224, 2050), (4224, 2500)])
def test_values_of_discarded_tokens_stay_out(gpu, monkeypatch, tmp_path, ctx, at, kv):
    """Values of tokens that were dropped again lie in the cache past a row's last position, in the same 16 bytes as its own:
    infinite ones there change nothing (the row has `at` + 1 positions)."""
    t = Tables(64, 5)
    t.v[ORDINARY, ::3] = 1e5 if kv == "f16" else 4e39  # (4e39: the product overflows float32, its weight does not)
    ids = np.random.default_rng(6).integers(0, ORDINARY, at + 2)
    m = t.load(monkeypatch, str(tmp_path / "t.gguf"), ctx=ctx, kv=kv)
    want = t.exact(ids, [at, at + 1])
    for n in (1, 2):
        print(f"case discarded values after {at} of {ctx} kv {kv} passes of {n}", flush=True)
        m.truncate(0)
        for i in range(0, at, 64):
            m.forward_batch(ids[i:min(i + 64, at)].tolist(), logits="none")
        m.forward_batch([ORDINARY] * 9, logits="none")
        m.truncate(at)
        got = np.concatenate([m.forward_batch(ids[i:i + n].tolist(), logits="all").copy() for i in range(at, at + 2, n)])
        assert np.abs(t.outputs(got, ids[at:]) - want).max() <= 1e-5 * np.abs(want).max(), n
    m.close()


@pytest.mark.parametrize("head_dim,kv", [(64, "f16"), (128, "f16"), (128, "f32")])
def test_rows_of_more_chunks_than_have_blocks_of_their_own(gpu, monkeypatch, tmp_path, head_dim, kv):
    """Rows on both sides of 16, 17 and 18 chunks (blocks then walk two of them), and short rows of the same large cache."""
    t = Tables(head_dim, 8)
    ids = np.random.default_rng(9).integers(0, IDS, 36870)
    m = t.load(monkeypatch, str(tmp_path / "t.gguf"), ctx=36900, kv=kv)
    spans = [(700, 716), (4090, 4106), (32760, 32776), (34810, 34826), (36854, 36870)]
    got = {}
    for n in (1, 5, 16):
        print(f"case more chunks than blocks head {head_dim} kv {kv} passes of {n}", flush=True)
        m.truncate(0)
        at = 0
        for a, b in spans:
            for i in range(at, a, 64):
                m.forward_batch(ids[i:min(i + 64, a)].tolist(), logits="none")
            rows = np.concatenate([m.forward_batch(ids[i:min(i + n, b)].tolist(), logits="all").copy() for i in range(a, b, n)])
            at = b
            want = t.exact(ids, range(a, b))
            assert np.abs(t.outputs(rows, ids[a:b]) - want).max() <= 1e-5 * np.abs(want).max(), (n, a)
            assert (rows.view(np.uint32) == got.setdefault(a, rows).view(np.uint32)).all(), (n, a)
    m.close()
