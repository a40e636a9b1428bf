"""The OK_Q4B GEMM over a token batch against one decode step per token, bit for
bit (exact mode: the GEMM's integer is the GEMV's): each of its forms, picked by
the weights' scales (few low digits, listed; many, a third digit; over 9
exponents, the per-block GEMM), and each built shape of the folded ones (row
and K groups, token tiles, K splits, rows past the last whole tile)."""
import numpy as np
import pytest

import spkv
from helpers import gemm_forms, prompt, write_scaled

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


# (share of the 32-column blocks scaled, by 2^-k, in which matrices): none beyond
# the random init's own; a listed share of deep low digits; more than the list
# takes; more in one matrix of a launch; and, up instead of down so that no scale
# is rounded to f16's smallest step, one beyond the digits in some row of each
# matrix that does not feed the residual twice
SPREADS = {"plain": (0.0, 0, None), "listed": (0.003, 7, None), "digit3": (0.2, 6, None), "mixed": (0.2, 6, ("attn_k", "ffn_up")),
           "per-block": (0.004, -9, ("attn_q", "attn_output", "ffn_gate", "ffn_down"))}
FORMS = {"plain": {2}, "listed": {2}, "digit3": {3}, "mixed": {2, 3}, "per-block": {0, 2}}


class Steps:
    """A model's K/V and logits by single steps."""

    def __init__(self, tmpdir, shape, spread, n):
        spm, spt, self.d = write_scaled(tmpdir, shape, *SPREADS[spread], max_context=1024)
        forms = gemm_forms(spm, self.d)
        assert set(forms.values()) == FORMS[spread], forms
        if spread == "per-block":
            assert all(f == 0 for t, f in forms.items() if t.split(".")[-1] in SPREADS[spread][2]), forms
        self.m = spkv.Model(spm, spt)
        self.s = spkv.Session(self.m, 1024)
        self.qm = spkv.l1().sp_session_qwen3_model(self.s.h)
        self.V, self.kvd = self.d["vocab"], self.d["n_kv_heads"] * self.d["head_dim"]
        self.pr = prompt(n, self.V, seed=3)
        self.one = spkv.Backend(self.qm, n + 1, exact=True, batch_prefill=False)
        self.one.prefill(self.pr)
        self.kv = [self.one.read_kv(l, 0, n, self.kvd) for l in range(self.d["n_layers"])]
        self.lg = {}

    def logits(self, n):
        if n not in self.lg:
            self.one.rewind(self.one.position() - n)
            self.lg[n] = np.zeros(self.V, np.float32)
            self.one.decode(int(self.pr[0]), self.lg[n])
            self.one.rewind(1)
            self.one.prefill(self.pr[n:])              # the rows the step overwrote
        return self.lg[n]

    def check(self, n, shape=(0, 0, 0)):
        b = spkv.Backend(self.qm, len(self.pr) + 1, exact=True)
        spkv.check(spkv.kv().sp_hipkv_set_gemm_shape(b.h, *shape), "sp_hipkv_set_gemm_shape")
        b.prefill(self.pr[:n])
        for l, (k, v) in enumerate(self.kv):
            kb, vb = b.read_kv(l, 0, n, self.kvd)
            assert np.array_equal(bits(kb), bits(k[:n])) and np.array_equal(bits(vb), bits(v[:n])), (shape, n, l)
        lg = np.zeros(self.V, np.float32)
        b.decode(int(self.pr[0]), lg)
        assert np.array_equal(bits(lg), bits(self.logits(n))), (shape, n)
        b.close()

    def close(self):
        self.one.close(); self.s.close(); self.m.close()


@pytest.mark.parametrize("spread", list(SPREADS))
@pytest.mark.parametrize("shape", ["gemma3-wide", "qwen3-g4", "qwen3-ragged"])
def test_prefill_equals_decode_steps(tmpdir_models, shape, spread):
    """Prompts of 1 to 141 tokens through the batched GEMMs, in the shapes they pick."""
    st = Steps(tmpdir_models, shape, spread, 141)
    for n in (1, 15, 16, 17, 33, 64, 65, 141):
        st.check(n)
    st.close()


# k_groups, token_tiles; 4 token tiles are built for two digits only
BUILT = [(1, 1), (1, 2), (1, 4), (2, 2), (2, 4), (4, 1), (4, 2), (8, 1)]


@pytest.mark.parametrize("spread", ["listed", "mixed"])
@pytest.mark.parametrize("shape", ["gemma3-wide", "qwen3-ragged"])
def test_every_built_shape_equals_decode_steps(tmpdir_models, shape, spread):
    """Each built (K groups, token tiles), whole and split: the wide model's 18 and
    34 128-column steps split up to 3 ways at 8 K groups, unevenly at most
    shapes; the ragged one's 2 to 10 leave K groups without any, and its q/k/v
    rows end within a tile.  1 to 512 tokens: one tile, part of one, part of a
    token group, a whole pass."""
    st = Steps(tmpdir_models, shape, spread, 512)
    for wk, tt in BUILT:
        for ks in (1, 2, 3, 4):
            if tt == 4 and spread == "mixed":          # refused at the launch, nothing run
                b = spkv.Backend(st.qm, 64, exact=True)
                assert spkv.kv().sp_hipkv_set_gemm_shape(b.h, wk, tt, ks) == 0
                assert spkv.kv().sp_hipkv_prefill(b.h, spkv.ptr(st.pr), 5) != 0 and b.position() == 0
                assert "shape that was set" in spkv.last_error()
                b.close()
                continue
            for n in (1, 17, 129, 512):
                st.check(n, (wk, tt, ks))
    st.close()


def test_set_gemm_shape_refuses_what_is_not_built(tmpdir_models):
    spm, spt, d = write_scaled(tmpdir_models, "qwen3-g4", 0.0, 0)
    m = spkv.Model(spm, spt)
    s = spkv.Session(m, 64)
    b = spkv.Backend(spkv.l1().sp_session_qwen3_model(s.h), 64, exact=True)
    for bad in ((3, 1, 1), (1, 3, 1), (8, 2, 1), (1, 1, 0), (1, 1, 17), (0, 1, 1), (-1, -1, -1)):
        assert spkv.kv().sp_hipkv_set_gemm_shape(b.h, *bad) != 0, bad
    assert spkv.kv().sp_hipkv_set_gemm_shape(b.h, 0, 0, 0) == 0
    b.close(); s.close(); m.close()


@pytest.mark.parametrize("spread", ["listed", "digit3"])
@pytest.mark.parametrize("n", [2, 16, 19])
def test_decode_batch_equals_single_steps(tmpdir_models, n, spread):
    """A batched step's logits rows are each session's own, bit for bit, in every
    built shape (the LM head's 2112 rows end within a 64- to 256-row tile)."""
    spm, spt, d = write_scaled(tmpdir_models, "qwen3-ragged", *SPREADS[spread])
    m = spkv.Model(spm, spt)
    s = spkv.Session(m, 64)
    qm = spkv.l1().sp_session_qwen3_model(s.h)
    V = d["vocab"]
    bs = [spkv.Backend(qm, 64, exact=True) for _ in range(n)]
    toks = prompt(n, V, seed=99)
    one = np.zeros((n, V), np.float32)
    for i, b in enumerate(bs):
        b.prefill(prompt(3 + i % 7, V, seed=i))
        b.decode(int(toks[i]), one[i])
        b.rewind(1)
    for shape in [(0, 0, 0)] + [(wk, tt, ks) for wk, tt in BUILT for ks in (1, 3) if tt < 4 or spread == "listed"]:
        spkv.check(spkv.kv().sp_hipkv_set_gemm_shape(bs[0].h, *shape), "sp_hipkv_set_gemm_shape")
        lg, nxt = spkv.Backend.decode_batch(bs, toks, V)
        for i, b in enumerate(bs):
            assert np.array_equal(bits(lg[i]), bits(one[i])) and int(nxt[i]) == int(one[i].argmax()), (shape, i)
            b.rewind(1)
    for b in bs:
        b.close()
    s.close(); m.close()
