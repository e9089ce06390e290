"""Prefill steps of many chunks at once, against the CPU oracle."""
import numpy as np
import pytest

import ana_amd
from ana_amd import ckpt
from ana_amd import config as cf

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


def _model(tmp_path, d, heads, arms, ctx=64, layers=4, f=None, vocab=258):
    c = cf.Config(vocab, ctx, d, f or 3 * d, layers, heads, arms, arms, arms)
    path = str(tmp_path / "m.ftc2")
    ckpt.write(path, c, ckpt.init_params(c, "normal", 3, std=0.05, trained=True))
    return c, path


@pytest.mark.parametrize("arms", [True, False])
@pytest.mark.parametrize("d,heads", [(64, 4), (128, 4), (256, 4)])
def test_exact_ragged_steps(oracle, tmp_path, d, heads, arms):
    """k_gla_serial and the batched attention (hd 16, 32, 64): sequences
    whose chunks end around the serial wave's token blocks (1, 11, 12, 13,
    24, 25, 63 tokens), fed together and then again past the ring's wrap;
    states and logits bit for bit."""
    c, path = _model(tmp_path, d, heads, arms)
    m = oracle.Model(path)
    lens = [1, 11, 12, 13, 24, 25, 63]
    r = np.random.RandomState(d + heads)
    first = [r.randint(0, c.vocab, n).astype(np.uint32) for n in lens]
    more = [r.randint(0, c.vocab, 30 - 3 * i).astype(np.uint32) for i in range(len(lens))]
    seqs = [3, 0, 6, 1, 5, 2, 4]
    print(f"case exact ragged d {d} heads {heads} arms {arms}", flush=True)
    with ana_amd.Decoder(path, max_seqs=7, prefill_chunk=32) as dec:
        dec.feeds_n(seqs, [0] * 7, first)
        dec.feeds_n(seqs, lens, more)
        lg = dec.logits(seqs)
        for i, s in enumerate(seqs):
            st = oracle.State(m)
            st.feeds(0, np.concatenate([first[i], more[i]]))
            for l in range(c.layers):
                assert np.array_equal(bits(dec.state(s, l)), bits(st.layer(l))), (i, l)
            assert np.array_equal(bits(lg[i]), bits(st.logits())), i


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# (d, heads, MLP, sequences, tokens of the longest): the split tiles' remainders (rows
# past a 16-, 64- and 128-row tile, 16-row weight tiles past the last full
# one, 2 to 64 k steps, odd numbers among them) and, at the 115M's widths, each tile
# shape, plain and SiLU (test_capacity.test_split_tiles_covered)
SPLIT_CASES = [(64, 4, 192, 2, 70), (128, 4, 160, 3, 48), (256, 4, 1024, 5, 60), (256, 4, 352, 8, 65),
               (768, 12, 2048, 9, 115), (768, 12, 2048, 10, 121), (768, 12, 2048, 17, 125), (768, 12, 2048, 64, 128)]


def split_lens(n, plen):
    return [max(1, plen - 3 * (i % 5)) for i in range(n)]


@pytest.mark.parametrize("d,heads,f,n,plen", SPLIT_CASES)
def test_split_products(tmp_path, d, heads, f, n, plen):
    """fast_fp32 prefill steps of 128 rows or more (k_split3, k_gemm_x3)
    against the exact mode: every state and the logits. A product's parts
    leave out less than one fp32 rounding, so what differs is the order of
    fp32 sums: 1e-5 is about four times what k_gemm_big's fp32 products
    show."""
    c, path = _model(tmp_path, d, heads, True, ctx=256, layers=4 if d < 768 else 2, f=f, vocab=512)
    lens = split_lens(n, plen)
    r = np.random.RandomState(d + f + n)
    toks = [r.randint(0, c.vocab, k).astype(np.uint32) for k in lens]
    seqs = list(range(n))
    print(f"case split products d {d} f {f} rows {sum(lens)}", flush=True)
    out = []
    for mode in (ana_amd.FAST_FP32, ana_amd.EXACT_FP32):
        with ana_amd.Decoder(path, max_seqs=n, prefill_chunk=128, numerics=mode) as dec:
            dec.feeds_n(seqs, [0] * n, toks)
            out.append((dec.logits(seqs), [dec.state(s, l) for s in (0, n - 1) for l in range(c.layers + 1)]))
    assert _rel(out[0][0], out[1][0]) < 1e-5
    for a, b in zip(out[0][1], out[1][1]):
        assert _rel(a, b) < 1e-5
    with ana_amd.Decoder(path, max_seqs=n, prefill_chunk=128, numerics=ana_amd.FAST_FP32) as dec:
        ce = dec.score_n(seqs, [0] * n, toks)
    with ana_amd.Decoder(path, max_seqs=n, prefill_chunk=128) as dec:
        want = dec.score_n(seqs, [0] * n, toks)
    assert _rel(np.concatenate(ce), np.concatenate(want)) < 1e-5


def test_split_products_not_finite(tmp_path):
    """A row that is not finite stays its own: its logits are NaN, as the
    exact mode's, and the other sequences' what they are without it; a value
    in the last binade (which rounds to infinity in bf16) counts as it does
    in the exact mode."""
    c = cf.Config(512, 256, 64, 192, 1, 4, True, True, True)
    p = ckpt.init_params(c, "normal", 3, std=0.05, trained=True)
    p[5 * c.d] = np.inf                    # token 5's embedding
    p[6 * c.d] = np.float32(3.4e38)        # token 6's: its square overflows
    path = str(tmp_path / "m.ftc2")
    ckpt.write(path, c, p)
    toks = [np.full(64, 9, np.uint32) for _ in range(3)]
    with ana_amd.Decoder(path, max_seqs=3, prefill_chunk=64, numerics=ana_amd.FAST_FP32) as dec:
        dec.feeds_n([0, 1, 2], [0] * 3, toks)
        want = dec.logits([0, 1, 2])
        for q in range(3):
            dec.reset(q)
        toks[1][-1] = 5
        toks[2][-1] = 6
        dec.feeds_n([0, 1, 2], [0] * 3, toks)
        got = dec.logits([0, 1, 2])
    with ana_amd.Decoder(path, max_seqs=3, prefill_chunk=64) as dec:
        dec.feeds_n([0, 1, 2], [0] * 3, toks)
        exact = dec.logits([0, 1, 2])
    fin = np.delete(np.arange(c.vocab), [5, 6])   # (the tied head has those rows too)
    got, want, exact = got[:, fin], want[:, fin], exact[:, fin]
    assert np.isfinite(want).all() and np.array_equal(bits(got[0]), bits(want[0]))
    assert np.isnan(got[1]).all() and np.isnan(exact[1]).all()
    assert np.array_equal(np.isnan(got[2]), np.isnan(exact[2]))


@pytest.mark.parametrize("chunk", [1, 16, 64])
def test_exact_steps_over_the_wrap(oracle, tmp_path, chunk):
    """step_chunk's steps: a step's chunk runs up to the ring's wrap (64
    slots) whatever the context's chunk, and keeps to it past the wrap; one
    sequence, then three at once from different positions; bit for bit."""
    c, path = _model(tmp_path, 64, 4, True)
    m = oracle.Model(path)
    r = np.random.RandomState(chunk)
    toks = [r.randint(0, c.vocab, k).astype(np.uint32) for k in (150, 40, 23)]
    more = [r.randint(0, c.vocab, k).astype(np.uint32) for k in (9, 31, 41)]
    print(f"case exact steps over the wrap, chunk {chunk}", flush=True)
    with ana_amd.Decoder(path, max_seqs=3, prefill_chunk=chunk) as dec:
        for i in range(3):
            dec.feeds(i, 0, toks[i])
        dec.feeds_n([2, 0, 1], [23, 150, 40], [more[2], more[0], more[1]])
        for i in range(3):
            st = oracle.State(m)
            st.feeds(0, np.concatenate([toks[i], more[i]]))
            for l in range(c.layers):
                assert np.array_equal(bits(dec.state(i, l)), bits(st.layer(l))), (i, l)
            assert np.array_equal(bits(dec.logits([i])[0]), bits(st.logits())), i


@pytest.mark.parametrize("n,plen", [(1, 300), (3, 300), (15, 280), (16, 300), (40, 260)])
def test_fast_steps(tmp_path, n, plen):
    """step_chunk's longer chunks in fast_fp32, on both sides of its rules
    (the GLA scan for fewer than 16 sequences, chunks of at most 256 tokens
    from there, more rows than a step holds) against the exact mode, as
    test_split_products holds them."""
    c, path = _model(tmp_path, 64, 4, True, ctx=512, f=192)
    r = np.random.RandomState(n)
    toks = [r.randint(0, c.vocab, plen - i % 7).astype(np.uint32) for i in range(n)]
    seqs = list(range(n))
    print(f"case fast steps n {n}", flush=True)
    out = []
    for mode in (ana_amd.FAST_FP32, ana_amd.EXACT_FP32):
        with ana_amd.Decoder(path, max_seqs=n, numerics=mode) as dec:
            dec.feeds_n(seqs, [0] * n, toks)
            out.append((dec.logits(seqs), [dec.state(s, l) for s in (0, n - 1) for l in range(c.layers + 1)]))
    assert _rel(out[0][0], out[1][0]) < 1e-5
    for a, b in zip(out[0][1], out[1][1]):
        assert _rel(a, b) < 1e-5


@pytest.mark.parametrize("n,chunk,plen,ctx", [(1, 64, 300, 512), (3, 32, 200, 512), (15, 8, 60, 64), (2, 48, 150, 64),
                                              (16, 64, 100, 512), (1, 128, 300, 256)])
def test_bf16_steps_keep_the_chunk(tmp_path, n, chunk, plen, ctx):
    """In bf16 a step's rows decide what is rounded (under 128 rows the first
    block stays in fp32), so for any number of sequences a step is a chunk of
    each: prompts (and scored windows) in one call are to the bit what they
    are a chunk a call, before the ring's wrap and over it."""
    c, path = _model(tmp_path, 256, 4, True, ctx=ctx, f=512)
    r = np.random.RandomState(n + chunk)
    toks = [r.randint(0, c.vocab, plen - i % 7).astype(np.uint32) for i in range(n)]
    seqs = list(range(n))
    print(f"case bf16 steps n {n} chunk {chunk} ctx {ctx}", flush=True)

    def read(dec):
        return [dec.logits(seqs)] + [dec.state(s, l) for s in (0, n - 1) for l in range(c.layers + 1)]

    with ana_amd.Decoder(path, max_seqs=n, prefill_chunk=chunk, numerics=ana_amd.BF16) as dec:
        dec.feeds_n(seqs, [0] * n, toks)
        whole = read(dec)
        for q in seqs:
            dec.reset(q)
        ce = dec.score_n(seqs, [0] * n, toks)
        for q in seqs:
            dec.reset(q)
        for t0 in range(0, plen, chunk):
            on = [q for q in seqs if toks[q].size > t0]
            dec.feeds_n(on, [t0] * len(on), [toks[q][t0:t0 + chunk] for q in on])
        parts = read(dec)
        for q in seqs:
            dec.reset(q)
        pce = [[] for _ in seqs]
        for t0 in range(0, plen - 1, chunk):
            on = [q for q in seqs if toks[q].size - 1 > t0]
            for q, v in zip(on, dec.score_n(on, [t0] * len(on), [toks[q][t0:t0 + chunk + 1] for q in on])):
                pce[q].append(v)
    for a, b in zip(whole, parts):
        assert np.array_equal(bits(a), bits(b))
    for a, b in zip(ce, pce):
        assert np.array_equal(bits(a), bits(np.concatenate(b)))


@pytest.mark.parametrize("arms", [True, False])
@pytest.mark.parametrize("d,heads,f", [(64, 4, 192), (128, 4, 352), (256, 4, 1024)])
def test_exact_single_feeds(oracle, tmp_path, d, heads, f, arms):
    """One sequence's feeds (the persistent launch without its head; hd 16,
    32, 64) from an empty slot to past the ring's wrap, between greedy loops,
    feeds of two sequences and a reset; states, logits and picks bit for
    bit, a sequence beside them untouched."""
    c, path = _model(tmp_path, d, heads, arms, ctx=32, f=f)
    m = oracle.Model(path)
    r = np.random.RandomState(d + arms)
    print(f"case exact single feeds d {d} arms {arms}", flush=True)
    with ana_amd.Decoder(path, max_seqs=3) as dec:
        st = {q: oracle.State(m) for q in (0, 1, 2)}
        pos = {0: 0, 1: 0, 2: 0}

        def feed(seqs):
            toks = [int(r.randint(0, c.vocab)) for _ in seqs]
            dec.feed(seqs, [pos[q] for q in seqs], toks)
            for q, t in zip(seqs, toks):
                st[q].feed(pos[q], t)
                pos[q] += 1

        def check(q):
            for l in range(c.layers):
                assert np.array_equal(bits(dec.state(q, l)), bits(st[q].layer(l))), (q, l, pos[q])
            assert np.array_equal(bits(dec.logits([q])[0]), bits(st[q].logits())), (q, pos[q])
            assert int(dec.top([q])[0]) == int(oracle.top(st[q].logits()))

        feed([1])
        check(1)
        for k in range(34):                  # the ring's wrap at 32
            feed([2])
            if k in (0, 1, 15, 31, 32, 33):
                check(2)
        feed([0, 2])
        feed([2])
        t = int(oracle.top(st[2].logits()))
        ids = dec.generate([2], [pos[2]], [t], 3)
        for g in np.asarray(ids).reshape(-1):
            st[2].feed(pos[2], t)
            pos[2] += 1
            t = int(oracle.top(st[2].logits()))
            assert int(g) == t
        feed([2])
        check(2)
        check(0)
        check(1)
        dec.reset(2)
        st[2], pos[2] = oracle.State(m), 0
        feed([2])
        check(2)


@pytest.mark.parametrize("arms", [True, False])
@pytest.mark.parametrize("d,heads,f", [(64, 4, 192), (128, 4, 352), (256, 4, 1024)])
@pytest.mark.parametrize("plen", [20, 45])
def test_exact_feed_after_a_timeout(oracle, tmp_path, monkeypatch, d, heads, f, arms, plen):
    """A feed whose launch counts as timed out (a limit of 0 ms) is undone
    and fed by the kernels (before the ring's wrap at 32 and past it), and so
    are the ones after it; a loop's time-out is reported, and the reset
    sequence is a fresh one. States and logits bit for bit, a sequence beside
    it untouched."""
    c, path = _model(tmp_path, d, heads, arms, ctx=32, f=f)
    m = oracle.Model(path)
    r = np.random.RandomState(d + arms + plen)
    toks = r.randint(0, c.vocab, plen + 3).astype(np.uint32)
    monkeypatch.setenv("ANA_PERSIST_MS", "0")
    print(f"case exact feed after a time-out d {d} arms {arms} from {plen}", flush=True)
    with ana_amd.Decoder(path, max_seqs=2) as dec:
        st, beside = oracle.State(m), oracle.State(m)

        def check(q, want):
            for l in range(c.layers):
                assert np.array_equal(bits(dec.state(q, l)), bits(want.layer(l))), (q, l)
            assert np.array_equal(bits(dec.logits([q])[0]), bits(want.logits())), q

        dec.feeds(0, 0, toks[:9])
        beside.feeds(0, toks[:9])
        dec.feeds(1, 0, toks[:plen])
        st.feeds(0, toks[:plen])
        for k in range(plen, plen + 3):
            dec.feed([1], [k], [int(toks[k])])
            st.feed(k, int(toks[k]))
            check(1, st)
        with pytest.raises(ana_amd.AnaError, match="time limit"):
            dec.generate([1], [plen + 3], [5], 4)
        dec.reset(1)
        dec.feed([1], [0], [6])
        st = oracle.State(m)
        st.feed(0, 6)
        check(1, st)
        check(0, beside)


def test_exact_loops_after_many_feeds(oracle, tmp_path):
    """Greedy loops after as many single feeds as turn a 16-bit count of
    epochs around (three a feed): to the tag that the context's untouched
    keys have, and from a loop's second step to the next loop's first one.
    Picks and logits bit for bit."""
    c, path = _model(tmp_path, 64, 4, True, ctx=32)
    m = oracle.Model(path)
    with ana_amd.Decoder(path, max_seqs=1) as dec:
        for feeds in (21845, 21844):
            print(f"case loops after {feeds} feeds", flush=True)
            for k in range(feeds - 1):   # (and the one below)
                dec.feed([0], [k % 40], [k % c.vocab])
            dec.reset(0)
            st = oracle.State(m)
            dec.feed([0], [0], [7])
            st.feed(0, 7)
            t = int(oracle.top(st.logits()))
            want = [t]
            for k in range(5):
                st.feed(1 + k, want[-1])
                want.append(int(oracle.top(st.logits())))
            got = dec.generate([0], [1], [t], 5)
            assert np.asarray(got).reshape(-1).tolist() == want[1:], feeds
            assert np.array_equal(bits(dec.logits([0])[0]), bits(st.logits())), feeds


@pytest.mark.parametrize("d,heads,ctx", [(64, 4, 5), (128, 4, 64), (768, 12, 2048)])
def test_reset_clears_one_sequence(tmp_path, d, heads, ctx):
    """k_reset (hd 16, 32, 64; states of less than a workgroup's stores and
    more than the grid's): the sequence's states and residual row are what a
    slot never fed has, its neighbours' are what they were, to the bit."""
    c, path = _model(tmp_path, d, heads, True, ctx=ctx, f=2 * d)
    print(f"case reset d {d} ctx {ctx}", flush=True)
    with ana_amd.Decoder(path, max_seqs=4, prefill_chunk=32) as dec:
        fresh = [dec.state(3, l) for l in range(c.layers + 1)]
        assert not any(a.any() for a in fresh)
        for q in (0, 1, 2):
            dec.feeds(q, 0, np.arange(q, q + ctx // 2 + 3, dtype=np.uint32) % c.vocab)
        before = {q: [dec.state(q, l) for l in range(c.layers + 1)] for q in (0, 2)}
        assert all(a.any() for a in (dec.state(1, l) for l in range(c.layers + 1)))
        dec.reset(1)
        for l in range(c.layers + 1):
            assert np.array_equal(bits(dec.state(1, l)), bits(fresh[l])), l
            for q in (0, 2):
                assert np.array_equal(bits(dec.state(q, l)), bits(before[q][l])), (q, l)
