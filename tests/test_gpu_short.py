"""Short batches (2 .. 64 tokens, csrc/lv_short.h; to 256, csrc/lv_mid.h) of LLaMA models against the CPU checker: every edge of the token tiles (16) and of
the kernels' limit, head sizes 32, 64 and 128, both weight types, K slices, contexts in front of the batch.

Tolerance: the one the path is specified with (test_gpu_model.py): 1e-2 and 1e-3 of the largest logit."""
import numpy as np
import pytest

import ggjt_builder as gb

pytestmark = pytest.mark.gpu

SHAPES = {
    "q4_32": ("Q4_0", dict(vocab=512, dim=384, heads=12, layers=2, ff=640)),
    "q4_64": ("Q4_0", dict(vocab=500, dim=512, heads=8, layers=2, ff=1408)),      # a vocabulary that 16 does not divide
    "q4_128": ("Q4_0", dict(vocab=512, dim=2048, heads=16, layers=1, ff=5504)),   # rows of 43 chunks: the waves' shares differ
    "q8_64": ("Q8_0", dict(vocab=512, dim=384, heads=6, layers=2, ff=896)),
    "q8_128": ("Q8_0", dict(vocab=512, dim=2048, heads=16, layers=1, ff=5504)),
}
# wide enough for four and six row tiles a workgroup, as many as 64 tokens and LDS allow at a time
WIDE = {
    "q4_wide": ("Q4_0", dict(vocab=512, dim=4096, heads=32, layers=1, ff=11008)),
    "q8_wide": ("Q8_0", dict(vocab=512, dim=4096, heads=32, layers=1, ff=11008)),
    "q4_wider": ("Q4_0", dict(vocab=512, dim=5120, heads=40, layers=1, ff=13824)),
    # a feed-forward at the limit of what goes to the kernel without LDS stages for 17 to 32 tokens: its largest row tiles
    "q4_tall": ("Q4_0", dict(vocab=512, dim=384, heads=12, layers=1, ff=8320)),
    "q8_tall": ("Q8_0", dict(vocab=512, dim=384, heads=6, layers=1, ff=5376)),
}
# six row tiles a workgroup on the way down, the last workgroup two: rows and statistics of part of a row group
RAGGED = {"q4_ragged": ("Q4_0", dict(vocab=512, dim=6656, heads=52, layers=1, ff=17920))}


@pytest.fixture(scope="module")
def models(lva, tmp_path_factory):
    d = tmp_path_factory.mktemp("short")
    out = {}
    for i, (name, (wtype, shape)) in enumerate({**SHAPES, **WIDE, **RAGGED}.items()):
        out[name] = str(d / f"{name}.ggml")
        lva.write_model(out[name], wtype=getattr(lva, "LV_" + wtype), seed=60 + i, **shape)
    for name in ("q4_64", "q8_64"):      # file version 1, whose block scales need fp32
        out[name + "_v1"] = str(d / f"{name}_v1.ggml")
        gb.convert_to_v1(out[name], out[name + "_v1"], jitter_seed=3)
    return out


def close(got, want):
    err = np.max(np.abs(got - want))
    assert err <= 1e-2 and err <= 1e-3 * np.max(np.abs(want)), (err, np.max(np.abs(want)))


CASES = [(name, b, n) for name in [*SHAPES, "q4_64_v1", "q8_64_v1"]
         for b, n in [(0, 2), (0, 16), (5, 17), (0, 33), (61, 3), (64, 48), (120, 64), (190, 65), (201, 49),
                       (1, 15), (2, 15), (49, 15), (50, 15), (200, 2), (239, 15)]]      # attention of up to 15 tokens: edges of its 16 and 64 positions
CASES += [(name, b, n) for name in RAGGED for b, n in [(0, 3), (3, 9)]]
CASES += [(name, b, n) for name in WIDE for b, n in [(0, 3), (70, 15), (0, 16), (0, 32), (9, 40), (0, 49), (130, 64)]]


@pytest.mark.parametrize("name,before,n", CASES)
def test_short_batch_matches_oracle(lva, orc, ctx, models, name, before, n):
    om = orc.Model(models[name])
    osess = orc.Session(om, 256)
    model = lva.Model(ctx, models[name])
    sess = lva.Session(model, 256)
    toks = lva.synth_tokens(before + n + 1, 3, om.hp["vocab"], seed=before + n)
    if before:
        osess.eval(toks[:before])
        sess.begin(toks[:before], 0)
        sess.wait()
        for layer in range(om.hp["layers"]):       # the batch under test starts from the checker's cache
            for which in (0, 1):
                sess.kv_write(layer, which, osess.kv(layer, which, before))
    want = osess.eval(toks[before:before + n])
    sess.begin(toks[before:before + n], before)
    close(sess.logits(), want)
    assert sess.argmax() == int(np.argmax(sess.logits()))
    for which in (0, 1):                           # its cache rows: at most an fp16 rounding apart in layer 0
        g, o = (s.kv(0, which, before + n)[before:].view(np.float16).astype(np.float32) for s in (sess, osess))
        assert np.max(np.abs(g - o)) <= np.max(np.abs(o)) * 2.0 ** -10
    want = osess.eval(toks[-1:])                   # ... which the next token reads
    sess.begin(toks[-1:], before + n)
    close(sess.logits(), want)
    sess.close(); model.close(); osess.close(); om.close()


@pytest.mark.parametrize("before,n", [(1900, 16), (1940, 33), (2040, 16), (2017, 31), (2100, 32), (2200, 33), (2300, 64), (2300, 15)])
def test_attention_of_short_steps_behind_long_contexts(lva, ctx, tmp_path, before, n):
    """one or two workgroups a CU, by the context's tiles a workgroup, on either side of where it changes; against the operator chain"""
    path = str(tmp_path / "forty.ggml")
    lva.write_model(path, wtype=lva.LV_Q8_0, seed=11, vocab=512, dim=1280, heads=40, layers=1, ff=1408)
    model = lva.Model(ctx, path)
    toks = lva.synth_tokens(before + n, 3, 512, seed=n)
    a, b = lva.Session(model, before + n), lva.Session(model, before + n)
    b.set_path(lva.PATH_KERNELS)
    a.begin(toks[:before], 0)
    a.wait()
    for which in (0, 1):
        b.kv_write(0, which, a.kv(0, which, before))
    for s in (a, b):
        s.keep_all_logits()
    a.begin(toks[before:], before)
    got = a.logits_rows(0, n)
    for i in range(n):
        b.begin(toks[before + i:before + i + 1], before + i)
        close(got[i], b.logits())
    a.close(); b.close(); model.close()


@pytest.mark.parametrize("rot,heads", [(32, 4), (64, 8), (128, 3)])
@pytest.mark.parametrize("before,n", [(63, 2), (64, 15), (800, 10), (800, 11), (1500, 2), (1500, 15)])
def test_parts_of_short_attention_put_together_by_the_last(lva, ctx, tmp_path, rot, heads, before, n):
    """two parts and the most there are, fewest and most tokens; two layers and two steps, so that a count left over would show.  Of heads of 128
    the last part to arrive adds up 10 tokens behind 800 rows, a launch of its own 11"""
    path = str(tmp_path / "heads.ggml")
    lva.write_model(path, wtype=lva.LV_Q4_0, seed=12, vocab=512, dim=rot * heads, heads=heads, layers=2, ff=512)
    model = lva.Model(ctx, path)
    total = before + 2 * n
    toks = lva.synth_tokens(total, 3, 512, seed=n)
    a, b = lva.Session(model, total), lva.Session(model, total)
    b.set_path(lva.PATH_KERNELS)
    a.begin(toks[:before], 0)
    a.wait()
    for layer in (0, 1):
        for which in (0, 1):
            b.kv_write(layer, which, a.kv(layer, which, before))
    for s in (a, b):
        s.keep_all_logits()
    for at in (before, before + n):
        a.begin(toks[at:at + n], at)
        got = a.logits_rows(0, n)
        for i in range(n):
            b.begin(toks[at + i:at + i + 1], at + i)
            close(got[i], b.logits())
    a.close(); b.close(); model.close()


# steps of 65 to 256 tokens (csrc/lv_mid.h), and what is left of a longer one: every edge of the token tiles and of the two groups of them
MIDDLE = [(name, 0, n) for name in ("q4_64", "q8_128") for n in (65, 80, 81, 96, 97, 128, 129, 160, 161, 192, 193, 256)]
MIDDLE += [(name, 37, n) for name in [*SHAPES, "q4_64_v1", "q8_64_v1"] for n in (70, 120, 170)]
MIDDLE += [("q4_64", 0, 513), ("q8_64", 3, 600), ("q4_wide", 0, 129), ("q8_wide", 5, 100), ("q4_wider", 0, 90), ("q4_wider", 0, 200)]


@pytest.mark.parametrize("name,before,n", MIDDLE)
def test_longer_step_matches_oracle(lva, orc, ctx, models, name, before, n):
    om = orc.Model(models[name])
    osess = orc.Session(om, 1024)
    model = lva.Model(ctx, models[name])
    sess = lva.Session(model, 1024)
    toks = lva.synth_tokens(before + n + 1, 3, om.hp["vocab"], seed=before + n)
    if before:
        osess.eval(toks[:before])
        sess.begin(toks[:before], 0)
        sess.wait()
        for layer in range(om.hp["layers"]):
            for which in (0, 1):
                sess.kv_write(layer, which, osess.kv(layer, which, before))
    want = osess.eval(toks[before:before + n])
    sess.begin(toks[before:before + n], before)
    close(sess.logits(), want)
    for which in (0, 1):
        g, o = (s.kv(0, which, before + n)[before:].view(np.float16).astype(np.float32) for s in (sess, osess))
        assert np.max(np.abs(g - o)) <= np.max(np.abs(o)) * 2.0 ** -10
    want = osess.eval(toks[-1:])                   # reads every cache row the step wrote
    sess.begin(toks[-1:], before + n)
    close(sess.logits(), want)
    sess.close(); model.close(); osess.close(); om.close()


@pytest.mark.parametrize("name,n", [("q4_64", 100), ("q8_64", 150)])
def test_every_row_of_a_longer_step(lva, ctx, models, name, n):
    """against a session whose path is set, which evaluates them as a batch in tiles of 128 tokens"""
    model = lva.Model(ctx, models[name])
    a, b = lva.Session(model, 256), lva.Session(model, 256)
    b.set_path(lva.PATH_GRAPH)
    toks = lva.synth_tokens(n, 3, 500, seed=n)
    rows = []
    for s in (a, b):
        s.keep_all_logits()
        s.begin(toks, 0)
        rows.append(s.logits_rows(0, n))
        assert np.array_equal(rows[-1][-1], s.logits())
    for i in range(n):
        close(rows[0][i], rows[1][i])
    a.close(); b.close(); model.close()


@pytest.mark.parametrize("name", ["q4_64", "q8_128"])
@pytest.mark.parametrize("n", [2, 31, 64])
def test_every_row_of_a_short_batch(lva, ctx, models, name, n):
    """lv_logits_read_rows against the same tokens one by one: both fp32, the cache rows rounded alike but for ties"""
    model = lva.Model(ctx, models[name])
    a, b = lva.Session(model, 128), lva.Session(model, 128)
    toks = lva.synth_tokens(n, 3, 500, seed=n)
    a.keep_all_logits()
    a.begin(toks, 0)
    rows = a.logits_rows(0, n)
    assert np.array_equal(rows[-1], a.logits())
    for i, t in enumerate(toks):
        b.begin([t], i)
        close(rows[i], b.logits())
    a.close(); b.close(); model.close()


@pytest.mark.parametrize("n", [2, 6, 15])
def test_a_set_path_takes_short_steps_too(lva, ctx, tmp_path, n):
    """token by token on the path that is set: the bits of the same tokens one by one; AUTO, on the kernels for short steps, close to them"""
    path = str(tmp_path / "wide.ggml")
    lva.write_model(path, wtype=lva.LV_Q8_0, seed=9, vocab=512, dim=4096, heads=32, layers=1, ff=11008)
    model = lva.Model(ctx, path)
    toks = lva.synth_tokens(n, 3, 512, seed=n)
    auto = lva.Session(model, 128)
    auto.begin(toks, 0)
    for p in (lva.PATH_PERSISTENT, lva.PATH_KERNELS, lva.PATH_GRAPH):
        a, b = lva.Session(model, 128), lva.Session(model, 128)
        a.set_path(p); b.set_path(p)
        a.begin(toks, 0)
        for i, t in enumerate(toks):
            b.begin([t], i)
            b.wait()
        assert np.array_equal(a.logits(), b.logits()), p
        close(auto.logits(), a.logits())
        a.close(); b.close()
    auto.close(); model.close()


@pytest.mark.parametrize("wtype,same", [("Q4_0", True), ("Q8_0", False)])
def test_two_tokens_of_a_wide_model(lva, ctx, tmp_path, wtype, same):
    """two launches of the persistent kernel read q4_0 in less time than one step of the kernels for short steps, q8_0 not"""
    path = str(tmp_path / "wide.ggml")
    lva.write_model(path, wtype=getattr(lva, "LV_" + wtype), seed=9, vocab=512, dim=4096, heads=32, layers=1, ff=11008)
    model = lva.Model(ctx, path)
    a, b = lva.Session(model, 128), lva.Session(model, 128)
    toks = lva.synth_tokens(2, 3, 512, seed=2)
    a.begin(toks, 0)
    for i, t in enumerate(toks):
        b.begin([t], i)
        b.wait()
    assert np.array_equal(a.logits(), b.logits()) == same
    close(a.logits(), b.logits())
    a.close(); b.close(); model.close()


def tensors(data):
    """name, type, elements and bytes of a version-3 file's tensors"""
    cur = 36
    for _ in range(int(data[8:12].view(np.uint32)[0])):
        cur += 8 + int(data[cur:cur + 4].view(np.int32)[0])
    while cur != len(data):
        dims, name_len, ftype = (int(v) for v in data[cur:cur + 12].view(np.uint32))
        count = int(np.prod(data[cur + 12:cur + 12 + 4 * dims].view(np.uint32)))
        name = data[cur + 12 + 4 * dims:cur + 12 + 4 * dims + name_len].tobytes().decode()
        cur = (cur + 12 + 4 * dims + name_len + 31) & ~31
        size = {0: 4 * count, 2: count // 32 * 18, 8: count // 32 * 34}[ftype]
        yield name, ftype, count, data[cur:cur + size]
        cur += size


def scaled_file(src, dst, powers):
    """a copy of a version-3 file with the blocks of some tensors multiplied by powers of two; powers: end of the name -> exponent"""
    data = np.fromfile(src, dtype=np.uint8)
    for name, _, count, payload in tensors(data):
        for end, e in powers.items():
            if name.endswith(end + ".weight"):
                d = payload.reshape(-1, len(payload) // (count // 32))
                d[:, :2] = np.ldexp(d[:, :2].copy().view(np.float16).astype(np.float32), e).astype(np.float16).view(np.uint8)
    data.tofile(dst)
    return dst


# feed-forward products of 1e5 and more, beyond fp16, and of 1e-6, where an fp16 pair has few bits left; the way down evens them out.
# Queries beyond fp16 on small keys; from 16 tokens on they are pairs, as in longer steps
LARGE, SMALL = {"w1": 12, "w3": 12, "w2": -8}, {"w1": -8, "w3": -8, "w2": 15}
MAGNITUDES = [("q4_64", LARGE, 16), ("q8_64", LARGE, 16), ("q4_64", SMALL, 16), ("q8_64", SMALL, 16),
              ("q4_64", {"wq": 19, "wk": -15}, 15), ("q8_64", {"wq": 17, "wk": -14}, 15)]


@pytest.mark.parametrize("name,powers,most", MAGNITUDES)
def test_short_batch_keeps_the_range_of_one_token_steps(lva, orc, ctx, models, tmp_path, name, powers, most):
    path = scaled_file(models[name], str(tmp_path / "scaled.ggml"), powers)
    om = orc.Model(path)
    model = lva.Model(ctx, path)
    for n in (2, 8, 9, 15, most):
        osess, a, b = orc.Session(om, 128), lva.Session(model, 128), lva.Session(model, 128)
        toks = lva.synth_tokens(n, 3, 500, seed=n)
        want = osess.eval(toks)
        a.begin(toks, 0)
        for i, t in enumerate(toks):
            b.begin([t], i)
            b.wait()
        assert np.isfinite(want).all()
        close(b.logits(), want)
        close(a.logits(), want)
        a.close(); b.close(); osess.close()
    model.close(); om.close()


@pytest.mark.parametrize("name", ["q4_32", "q8_64", "q4_128"])
@pytest.mark.parametrize("n", [2, 6, 15])
def test_a_token_beyond_fp16_does_not_reach_those_before_it(lva, ctx, models, tmp_path, name, n):
    """cache rows of infinities (and of NaN in the layer behind) in a step: the tokens that do not see them give the bits they give without"""
    path, wild = str(tmp_path / "wild.ggml"), 7
    data = np.fromfile(models[name], dtype=np.uint8)
    dim = SHAPES[name][1]["dim"]
    for tensor, ftype, _, payload in tensors(data):
        if tensor == "tok_embeddings.weight":
            assert ftype == 0
            table = payload.view(np.float32).reshape(-1, dim)
            table[:, 0] = 0
            table[wild] = np.eye(dim)[0]
        if tensor == "layers.0.attention_norm.weight":
            payload.view(np.float32)[0] = 1e8
    data.tofile(path)
    model = lva.Model(ctx, path)
    toks = np.array(lva.synth_tokens(n, 20, 480, seed=n), dtype=np.uint32)
    rows = []
    for change in (False, True):
        s = lva.Session(model, 128)
        s.keep_all_logits()
        if change:
            toks[n - 2 if n > 2 else 1] = wild
        s.begin(toks, 0)
        rows.append(s.logits_rows(0, n))
        if change:
            assert np.isinf(s.kv(0, 1, n).view(np.float16)).any()
        s.close()
    seen = n - 2 if n > 2 else 1
    assert np.isfinite(rows[0]).all()
    assert np.array_equal(rows[0][:seen], rows[1][:seen])
    model.close()
