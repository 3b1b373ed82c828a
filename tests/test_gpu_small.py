"""One token of a small model as one launch (lv_small.h) against the oracle and the operator chain: rows that fill tiles and rows that do not,
one and several blocks a lane, every head size, contexts on both sides of what the workgroup holds of the cache at once."""
import ctypes as C
import time

import numpy as np
import pytest

import ggjt_builder as gb

pytestmark = pytest.mark.gpu

ABS_TOL, REL_TOL = 1e-2, 1e-3       # of a whole evaluation in fp32 with fp16 cache rows, as in the other tests of whole models


def _check(got, want):
    err = np.max(np.abs(got - want))
    assert err <= ABS_TOL and err <= REL_TOL * np.max(np.abs(want)), (err, np.max(np.abs(want)))


# no width is a multiple of 128 where steps of several tokens are compared: those models have other kernels for such steps
SHAPES = {
    "one head, one block": dict(vocab=259, dim=32, heads=1, layers=1, ff=32),
    "three blocks a row": dict(vocab=500, dim=96, heads=3, layers=2, ff=224),
    "two columns a lane": dict(vocab=512, dim=256, heads=4, layers=2, ff=2080),
    "head of 128": dict(vocab=513, dim=256, heads=2, layers=3, ff=704),
    "sixteen heads": dict(vocab=4099, dim=512, heads=16, layers=2, ff=1376),
    "widest": dict(vocab=1000, dim=1024, heads=16, layers=2, ff=8160),
    "longest feed-forward": dict(vocab=600, dim=992, heads=31, layers=2, ff=8192),
    "more heads than tiles": dict(vocab=260, dim=1024, heads=32, layers=1, ff=64),
    "wide heads of 128": dict(vocab=1000, dim=1024, heads=8, layers=2, ff=8160),       # one workgroup a head would take longer: the chain
    "a block a workgroup": dict(vocab=512, dim=256, heads=8, layers=2, ff=2016),        # one workgroup less than there may be
    "workgroups without blocks": dict(vocab=8000, dim=128, heads=4, layers=2, ff=96),
    "widest with partial sums": dict(vocab=700, dim=288, heads=9, layers=2, ff=1792),
    "two blocks a workgroup": dict(vocab=512, dim=256, heads=4, layers=2, ff=4064),     # the last one has one
    "narrowest without": dict(vocab=700, dim=320, heads=5, layers=2, ff=864),
    "large vocabulary": dict(vocab=32000, dim=1024, heads=16, layers=1, ff=64),        # a quarter of the CUs would take longer
}
CHAIN = {"wide heads of 128", "large vocabulary"}


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("wtype", ["q4_0", "q8_0", "q4_0 version 1", "q8_0 table"])
def test_small_model_tokens_match_oracle_and_chain(lva, orc, ctx, tmp_path, shape, wtype):
    p, c = str(tmp_path / "m.ggml"), SHAPES[shape]
    table = {"1": lva.LV_Q4_0, "e": lva.LV_Q8_0}.get(wtype[-1], lva.LV_F32)       # of embeddings
    lva.write_model(p, wtype=lva.LV_Q8_0 if wtype.startswith("q8_0") else lva.LV_Q4_0, tok_type=table, seed=31, **c)
    if wtype.endswith("1"):
        gb.convert_to_v1(p, str(tmp_path / "v1.ggml"))
        p = str(tmp_path / "v1.ggml")
    om = orc.Model(p)
    osess = orc.Session(om, 512)
    model = lva.Model(ctx, p)
    one, other, chain = (lva.Session(model, 512) for _ in range(3))
    assert one.path() == lva.PATH_GRAPH
    chain.set_path(lva.PATH_GRAPH)
    toks = lva.synth_tokens(290, 3, c["vocab"], seed=2)
    pos, differ = 0, 0
    # alone, a step of several tokens, up to and across the borders of 64, 128 and 256 cache rows
    for n in (1, 1, 9, 1, 52, 1, 1, 61, 1, 1, 126, 1, 1, 1):
        step = toks[pos:pos + n]
        want = osess.eval(step)
        for s in (one, other, chain):           # sessions take turns on the device
            s.begin(step, pos)
        _check(one.logits(), want)
        _check(chain.logits(), want)
        assert np.array_equal(one.logits(), other.logits())
        differ += not np.array_equal(one.logits(), chain.logits())
        assert one.argmax() == int(np.argmax(one.logits()))
        pos += n
    assert (differ == 0) == (shape in CHAIN)    # which kernels ran: sums in another order round differently
    s = one
    s.keep_all_logits()
    s.begin(toks[:3], 0)
    rows = s.logits_rows(0, 3)
    assert np.array_equal(rows[2], s.logits())
    other.begin(toks[:1], 0)
    assert np.array_equal(rows[0], other.logits())
    for which in (0, 1):                        # cache rows of layer 0: the same inputs, sums in another order
        a, b = one.kv(0, which, 3), chain.kv(0, which, 3)
        assert np.mean(a != b) < 1e-2
    for s in (one, other, chain):
        s.close()
    model.close(); osess.close(); om.close()


def test_small_model_not_a_number_is_a_result_and_no_expired_wait(lva, ctx, tmp_path):
    """hand-overs wait until a value is there; the bit pattern that stands for `not there yet` is a NaN a model can hold"""
    p = str(tmp_path / "m.ggml")
    lva.write_model(p, wtype=lva.LV_Q4_0, seed=3, vocab=512, dim=256, heads=4, layers=2, ff=704)
    raw = np.fromfile(p, np.uint8)
    name = b"layers.0.ffn_norm.weight"
    at = (raw.tobytes().index(name) + len(name) + 31) // 32 * 32
    raw[at:at + 256 * 4] = 255
    raw.tofile(p)
    model = lva.Model(ctx, p)
    s = lva.Session(model, 128)
    for i in range(3):
        s.begin([5 + i], i)
        assert np.isnan(s.logits()).all()
    s.close(); model.close()


def test_small_models_sessions_run_beside_one_another(lva, ctx, tmp_path):
    """A launch takes a quarter of the CUs at most: four sessions' tokens take at most twice what one session's does where two of them
    share a hardware queue, four times it where each waits for the others' launches.  More sessions than that, each with its own tokens, get what each gets alone."""
    p, c = str(tmp_path / "m.ggml"), dict(vocab=1000, dim=768, heads=12, layers=8, ff=2048)
    lva.write_model(p, wtype=lva.LV_Q4_0, seed=8, **c)
    model = lva.Model(ctx, p)
    toks = [lva.synth_tokens(24, 3, c["vocab"], seed=i) for i in range(7)]
    alone, s = [], lva.Session(model, 64)
    for t in toks:
        for i in range(24):
            s.begin(t[i:i + 1], i)
            s.wait()
        alone.append(s.logits())
    s.close()
    several = [lva.Session(model, 64) for _ in toks]
    for i in range(24):
        for s, t in zip(several, toks):
            s.begin(t[i:i + 1], i)
        for s in several:
            s.wait()
    for s, want in zip(several, alone):
        assert np.array_equal(s.logits(), want)

    def fastest(sessions):
        times = []
        for _ in range(30):
            start = time.perf_counter()
            for s in sessions:
                s.begin(toks[0][:1], 24)
            for s in sessions:
                s.wait()
            times.append(time.perf_counter() - start)
        return min(times)
    assert fastest(several[:4]) < 3 * fastest(several[:1])
    for s in several:
        s.close()
    model.close()


def test_small_and_persistent_launches_of_one_context(lva, ctx, tmp_path):
    """the persistent kernel occupies every CU and runs behind all small launches, and these behind it"""
    small, large = dict(vocab=512, dim=256, heads=4, layers=2, ff=704), dict(vocab=512, dim=4096, heads=32, layers=2, ff=11008)
    models = []
    for i, c in enumerate((small, large)):
        lva.write_model(str(tmp_path / f"{i}.ggml"), wtype=lva.LV_Q4_0, seed=9, **c)
        models.append(lva.Model(ctx, str(tmp_path / f"{i}.ggml")))
    toks = lva.synth_tokens(40, 3, 512, seed=4)

    def decode(sessions):
        for i in range(len(toks)):
            for s in sessions:
                s.begin(toks[i:i + 1], i)
            out = [s.logits() for s in sessions]
        return out
    sessions = [lva.Session(models[k], 64) for k in (0, 1, 0, 0, 1, 0, 0, 0)]
    assert sessions[1].path() == lva.PATH_PERSISTENT
    want = [decode(sessions[k:k + 1])[0] for k in (0, 1)]
    for s, got in zip(sessions, decode(sessions)):
        assert np.array_equal(got, want[0 if s.model is models[0] else 1])
    for s in sessions:
        s.close()
    for m in models:
        m.close()


def _same_cache(dst, src, layers, n):
    for layer in range(layers):
        for which in (0, 1):
            dst.kv_write(layer, which, src.kv(layer, which, n))


def test_an_expired_wait_of_a_small_model_goes_unnoticed(lva, ctx, tmp_path):
    """with the poll bound at 1 every launch gives up; the call that waits evaluates the step on the operator chain, bit for bit what a session
    whose path is the chain gets, for every way of reading a step.  Two such steps in a row leave the session there, one does not"""
    p, c = str(tmp_path / "m.ggml"), dict(vocab=1000, dim=256, heads=4, layers=3, ff=704)
    lva.write_model(p, wtype=lva.LV_Q4_0, seed=12, **c)
    model = lva.Model(ctx, p)
    one, chain = lva.Session(model, 64), lva.Session(model, 64)
    chain.set_path(lva.PATH_KERNELS)
    toks = lva.synth_tokens(40, 3, c["vocab"], seed=6)
    pos = 0

    def step(n, read, limit):
        nonlocal pos
        _same_cache(one, chain, c["layers"], pos)
        one.set_wait_limit(limit)
        got = []
        for s in (one, chain):
            s.begin(toks[pos:pos + n], pos)
            got.append(read(s))
        pos += n
        return got

    def rows(s):
        return s.logits_rows(0, 2)

    def after_wait(s):
        s.wait()
        return s.logits()

    def timed(s):
        s.timer_start()
        s.timer_stop()
        return s.logits()
    differ = 0
    for n, read in ((1, lva.Session.logits), (3, lva.Session.logits), (1, lva.Session.argmax), (2, rows), (1, after_wait), (1, timed)):
        for s in (one, chain):
            s.keep_all_logits(read is rows)
        a, b = step(n, read, 1)                       # given up, evaluated again
        assert np.array_equal(a, b), read
        for s in (one, chain):
            s.keep_all_logits(False)
        a, b = step(1, lva.Session.logits, 0)         # not given up: the small models' kernel, whose sums round differently
        differ += not np.array_equal(a, b)
        _check(a, b)
    assert differ > 0
    for limit in (1, 1, 0, 0):                        # two in a row: the chain from then on
        a, b = step(1, lva.Session.logits, limit)
        assert np.array_equal(a, b)
    one.set_path(lva.PATH_AUTO)                       # another try
    assert any(not np.array_equal(*step(1, lva.Session.logits, 0)) for _ in range(4))
    one.close(); chain.close(); model.close()


def test_hand_over_buffers_of_ended_sessions_serve_models_of_other_sizes(lva, ctx, tmp_path):
    """they are never given back to the runtime: a process that goes through models of many sizes must not keep a pair for each.  17 to 30
    layers of 33 KB: 22 MB if each keeps its own, none beyond the first pair if they share one"""
    def free_memory():
        free, total = C.c_size_t(), C.c_size_t()
        assert lva.hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value
    before = None
    for layers in (30, *range(17, 30)):
        p = str(tmp_path / f"{layers}.ggml")
        lva.write_model(p, wtype=lva.LV_Q4_0, seed=3, vocab=259, dim=32, heads=1, layers=layers, ff=8192)
        model = lva.Model(ctx, p)
        s = lva.Session(model, 64)
        s.begin([5], 0)
        s.wait()
        s.close(); model.close()
        if before is None:
            before = free_memory()
    assert before - free_memory() < 8 << 20


@pytest.mark.parametrize("heads,border", [(2, 1024), (4, 2048)])
def test_a_small_models_session_moves_to_the_chain_behind_a_long_context(lva, ctx, tmp_path, heads, border):
    """One workgroup walks all cache rows of a head: from 131072 elements of them on the chain is faster.  On either side of that row, and in a
    step of several tokens that would cross it, with the same cache rows: bit for bit the chain's logits from there on, others before"""
    p, c = str(tmp_path / "m.ggml"), dict(vocab=700, dim=256, heads=heads, layers=2, ff=704)
    lva.write_model(p, wtype=lva.LV_Q8_0, seed=15, **c)
    model = lva.Model(ctx, p)
    one, chain = lva.Session(model, border + 64), lva.Session(model, border + 64)
    chain.set_path(lva.PATH_GRAPH)
    toks = lva.synth_tokens(border + 40, 3, c["vocab"], seed=7)
    chain.begin(toks[:border - 8], 0)
    chain.wait()
    for pos in range(border - 8, border - 2):
        chain.begin(toks[pos:pos + 1], pos)
        chain.wait()
    fresh, differ = True, {True: 0, False: 0}
    for pos, n in ((border - 2, 1), (border - 1, 1), (border - 1, 3), (border, 1), (border + 1, 1), (border - 2, 2), (border - 2, 3), (border + 1, 5)):
        _same_cache(one, chain, c["layers"], border - 2 if fresh else pos)
        fresh = False
        for s in (one, chain):
            s.begin(toks[pos:pos + n], pos)
        a, b = one.logits(), chain.logits()
        _check(a, b)
        differ[pos + n <= border] += not np.array_equal(a, b)
    assert differ[True] > 0 and differ[False] == 0
    one.close(); chain.close(); model.close()
