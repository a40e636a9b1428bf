"""The OK_Q4B GEMM over a token batch, at the edges of its dispatch: 16-token
tiles, token groups and K splits, and the scale spreads that pick its three
paths (few low digits, listed; many, a third digit; over 9 exponents, the
per-block GEMM)."""
import numpy as np
import pytest

import spkv
from helpers import prompt, write_scaled

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


# (share of the 32-column blocks scaled down, by 2^-k): none beyond the random
# init's own; a listed share of deep low digits; more than the list takes; one
# beyond the digits
SPREADS = {"plain": (0.0, 0), "listed": (0.003, 7), "digit3": (0.2, 6), "per-block": (0.05, 12)}


@pytest.mark.parametrize("spread", list(SPREADS))
@pytest.mark.parametrize("shape", ["gemma3-wide", "qwen3-g4"])
def test_prefill_equals_decode_steps(tmpdir_models, shape, spread):
    """Prompts of 1 to 141 tokens through the batched GEMMs leave the K/V and
    logits of one decode step per token, bit for bit (exact mode: the GEMM's
    integer is the GEMV's, whatever its digits, tiles and splits)."""
    spm, spt, d = write_scaled(tmpdir_models, shape, *SPREADS[spread])
    m = spkv.Model(spm, spt)
    s = spkv.Session(m, 256)
    qm = spkv.l1().sp_session_qwen3_model(s.h)
    V, kvd = d["vocab"], d["n_kv_heads"] * d["head_dim"]
    one = spkv.Backend(qm, 256, exact=True, batch_prefill=False)
    pr = prompt(141, V, seed=3)
    one.prefill(pr)
    ref = [one.read_kv(l, 0, 141, kvd) for l in range(d["n_layers"])]
    lg0, lg1 = np.zeros(V, np.float32), np.zeros(V, np.float32)
    for n in (1, 15, 16, 17, 33, 64, 65, 141):
        b = spkv.Backend(qm, 256, exact=True)
        b.prefill(pr[:n])
        for l, (k, v) in enumerate(ref):
            kb, vb = b.read_kv(l, 0, n, kvd)
            assert np.array_equal(bits(kb), bits(k[:n])) and np.array_equal(bits(vb), bits(v[:n])), (n, l)
        assert one.rewind(one.position() - n) == 0
        one.decode(int(pr[0]), lg0)
        b.decode(int(pr[0]), lg1)
        assert np.array_equal(bits(lg0), bits(lg1)), n
        b.close()
        one.rewind(1)
        one.prefill(pr[n:])                            # the rows the step overwrote
    one.close(); s.close(); m.close()


@pytest.mark.parametrize("n", [2, 16, 19])
def test_decode_batch_equals_single_steps(tmpdir_models, n):
    """A batched step's logits rows (the LM head's GEMM: rows not a multiple of
    the row tiles' groups) are each session's own, bit for bit."""
    spm, spt, d = write_scaled(tmpdir_models, "qwen3-g4", 0.2, 6)
    m = spkv.Model(spm, spt)
    s = spkv.Session(m, 64)
    qm = spkv.l1().sp_session_qwen3_model(s.h)
    V = d["vocab"]
    bs = [spkv.Backend(qm, 64, exact=True) for _ in range(n)]
    for i, b in enumerate(bs):
        b.prefill(prompt(3 + i % 7, V, seed=i))
    toks = prompt(n, V, seed=99)
    lg, _ = spkv.Backend.decode_batch(bs, toks, V)
    one = np.zeros(V, np.float32)
    for i, b in enumerate(bs):
        b.rewind(1)
        b.decode(int(toks[i]), one)
        assert np.array_equal(bits(lg[i]), bits(one)), i
        b.close()
    s.close(); m.close()
