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
