"""The buffers that batched calls of one model lease from each other: a call
with short contexts may take the set of one with long contexts, and what it adds
to that set serves the long ones afterwards."""
import threading

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


def test_float_prefill_does_not_depend_on_the_set(tmpdir_models):
    """A float prefill's position splits come from its own handle: the same bits
    on a set of its own and on the larger one another session left."""
    name, n = "gemma3-tiny", 600
    spm, spt = model_files(tmpdir_models, name, max_context=4160)
    V, NL = SMALL[name]["vocab"], SMALL[name]["n_layers"]
    kvd = SMALL[name]["n_kv_heads"] * SMALL[name]["head_dim"]
    out = []
    for larger in (False, True):
        m = spkv.Model(spm, spt)
        s = spkv.Session(m, 64)
        qm = spkv.l1().sp_session_qwen3_model(s.h)
        big = spkv.Backend(qm, 4160)
        if larger:
            big.prefill(prompt(70, V, seed=1))
        b = spkv.Backend(qm, 640)
        b.prefill(prompt(n, V, seed=2))
        out.append([b.read_kv(l, 0, n, kvd) for l in range(NL)])
        b.close(); big.close(); s.close(); m.close()
    for l, ((k0, v0), (k1, v1)) in enumerate(zip(*out)):
        assert np.array_equal(k0.view(np.uint32), k1.view(np.uint32)) and np.array_equal(v0.view(np.uint32), v1.view(np.uint32)), l


def test_calls_of_several_threads_modes_and_lengths(tmpdir_models):
    """Prefills and batched steps of handles with their own pmax and mode, from
    four threads at once on one model's sets, leave the bits of the same calls
    one after another."""
    name = "gemma3-w200"
    spm, spt = model_files(tmpdir_models, name, max_context=2048)
    V, NL = SMALL[name]["vocab"], SMALL[name]["n_layers"]
    kvd = SMALL[name]["n_kv_heads"] * SMALL[name]["head_dim"]
    m = spkv.Model(spm, spt)
    s = spkv.Session(m, 64)
    qm = spkv.l1().sp_session_qwen3_model(s.h)
    jobs = [(1600, True, 700), (300, False, 280), (640, False, 600), (64, True, 50)]

    def work(i, reps):
        pmax, exact, n = jobs[i]
        bs = [spkv.Backend(qm, pmax, exact=exact) for _ in range(2)]
        pr, toks = prompt(n, V, seed=40 + i), prompt(2, V, seed=50 + i)
        out = []
        for _ in range(reps):
            for b in bs:
                b.prefill(pr)
            lg, nxt = spkv.Backend.decode_batch(bs, toks, V)
            out.append([lg, nxt] + [x for l in range(NL) for x in bs[1].read_kv(l, 0, n, kvd)])
            for b in bs:
                b.rewind(n + 1)
        for b in bs:
            b.close()
        return out

    want = [work(i, 1)[0] for i in range(len(jobs))]
    got, errs = [None] * len(jobs), []

    def run(i):
        try:
            got[i] = work(i, 4)
        except Exception as e:                          # shown below
            errs.append((i, e))

    th = [threading.Thread(target=run, args=(i,)) for i in range(len(jobs))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errs, errs
    for i, reps in enumerate(got):
        for r, o in enumerate(reps):
            for j, (x, y) in enumerate(zip(o, want[i])):
                assert np.array_equal(x.view(np.uint32), y.view(np.uint32)), (i, r, j)
    s.close(); m.close()
