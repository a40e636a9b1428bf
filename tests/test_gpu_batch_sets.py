"""The buffers that batched calls of one model lease from each other: a call
with short contexts may take the set of one with long contexts, and what it adds
to that set serves the long ones afterwards."""
import numpy as np
import pytest

import spkv
from helpers import SMALL, model_files, prompt

pytestmark = pytest.mark.gpu


def test_a_short_batch_leaves_room_for_long_sessions(tmpdir_models):
    """A 4160-position session prefills, a batch of 64-position sessions steps on
    the set it gave back, then 64 sessions of 2061 to 2100 positions step: 5
    512-position chunks each, 320 work items (a list sized by the 64-position
    sessions holds 256).  Every row is its session's own single step, bit for
    bit, and again on the same set."""
    name, pmax, n = "qwen3-hd128", 4160, 64
    spm, spt = model_files(tmpdir_models, name, max_context=pmax)
    m = spkv.Model(spm, spt)
    s = spkv.Session(m, 64)
    qm = spkv.l1().sp_session_qwen3_model(s.h)
    V = SMALL[name]["vocab"]
    long = spkv.Backend(qm, pmax, exact=True)
    long.prefill(prompt(2100, V, seed=1))
    short = [spkv.Backend(qm, 64, exact=True) for _ in range(2)]
    for i, b in enumerate(short):
        b.prefill(prompt(5 + i, V, seed=2))
    spkv.Backend.decode_batch(short, prompt(2, V, seed=3), V)
    bs = [long.fork() for _ in range(n)]
    one = np.zeros(V, np.float32)
    for k in range(2):
        toks = prompt(n, V, seed=10 + k)
        for i, b in enumerate(bs):
            b.rewind(b.position() - (2060 + i % 40))
        lg, nxt = spkv.Backend.decode_batch(bs, toks, V)
        for i, b in enumerate(bs):
            b.rewind(1)
            b.decode(int(toks[i]), one)
            assert np.array_equal(lg[i].view(np.uint32), one.view(np.uint32)), (k, i)
            assert int(nxt[i]) == int(one.argmax()), (k, i)
    for b in bs + short + [long]:
        b.close()
    s.close(); m.close()
