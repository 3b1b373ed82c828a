"""The choice of experts: equal router rows tie to the last bit and the lower index wins, in one-token steps and in batches; on both
sides of 64 experts, where the choice of a token takes another form.

Small integers as embeddings, norm weights of one and router rows that come in equal pairs: an odd number of experts a token cuts a
pair.  The plain evaluation chooses by the same rule (choose_experts); a wrong pick is an error of order one.

And the inputs of one-token products, on both sides of the sizes up to which they are held in registers."""
import time

import numpy as np
import pytest

import block_builder as bb
import block_device
import block_oracle as bo
import zedenex_builder as zb
import zedenex_oracle as zo
from block_device import rel, tokens_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("experts,top,width", [(2, 1, 40), (6, 3, 640), (63, 5, 40), (64, 7, 1100), (65, 7, 40), (130, 9, 640)])
def test_equal_experts_tie(lva, ctx, experts, top, width):
    cfg = bb.config(width=width, layers=[bb.layer(experts=experts, top=top, ff=24)])
    W = bb.weights(cfg, seed=experts)
    for n in ("left", "right"):
        W[f"l0.mix.{n}.o"][:] = 0
    r = W["l0.mlp.router"]
    r[1::2] = r[0:experts - 1:2][: len(r[1::2])]
    toks = tokens_for(cfg, 40, 3)
    F = bb.as_float(W)
    h = bo.rms_norm(F["embed"][toks], F["l0.norm2"], cfg["norm"]["eps"])
    z = np.sort(h @ F["l0.mlp.router"].T, axis=1)[:, ::-1]
    cut = z[:, :-1] - z[:, 1:]                       # keep tokens whose choice is a tie inside a pair or clear
    near = cut[:, top - 1] if top < experts else np.ones(len(toks))
    toks = toks[(near < 1e-12) | (near > 0.05)]
    assert len(toks) > 10 and (near < 1e-12).sum() > 5
    want = bo.forward(toks, F, cfg)[0]
    with block_device.Device(lva, bb.upload(ctx, cfg, W, lva.LV_F32), 512) as d:
        for c in ((1000,), (1,), (16, 3)):
            assert rel(d.run(toks, c), want) < 2e-4, c


# What a one-token product's input is made of is held in registers up to a size, and read late behind it: on both sides of the 4096
# columns of a norm, 4096 attention outputs, 32 recurrent heads of 128 columns, and experts' down projections of 12288 columns together
WIDE = [
    (4160, dict(left=bb.attn(heads=2, kv_heads=1, dim=16)), dict(experts=3, top=2, ff=40)),
    (2112, dict(left=bb.attn(heads=33, kv_heads=3, dim=128, chunk=0)), dict(experts=5, top=4, ff=1100)),
    (48, dict(right=bb.delta(heads=34, kv_heads=17, dim=12, vdim=128)), dict(experts=2, top=1, ff=1030)),
    (72, dict(right=bb.delta(heads=36, kv_heads=4, dim=12, vdim=20)), dict(experts=7, top=6, ff=2060)),
    (64, dict(right=bb.delta(heads=3, kv_heads=3, dim=8, vdim=130)), dict(experts=0)),
]


@pytest.mark.parametrize("width,mix,ff", WIDE)
def test_inputs_beyond_the_early_part(lva, ctx, width, mix, ff):
    cfg = bb.config(width=width, layers=[bb.layer(**mix, **ff)])
    W = bb.weights(cfg, seed=width)
    toks = tokens_for(cfg, 20, 1)
    want = bo.forward(toks, bb.as_float(W), cfg)[0]
    with block_device.Device(lva, bb.upload(ctx, cfg, W, lva.LV_F32), 512) as d:
        assert rel(d.run(toks, (1,)), want) < 2e-4


# a read-out normed in parts: a wave's first task in registers (four quads a lane), the rest of it and further tasks late; parts that are no
# multiple of four
@pytest.mark.parametrize("heads,vdim,groups", [(64, 130, 1), (40, 130, 2), (40, 130, 8), (36, 64, 9), (24, 96, 36), (6, 7, 2)])
def test_grouped_input(lva, ctx, heads, vdim, groups):
    cfg = zb.config(width=52, streams=2, layers=[zb.layer(zb.ssm(heads=heads, groups=2, state=16, vdim=vdim, norm_groups=groups), 0)])
    W = zb.weights(cfg, seed=heads + groups)
    toks = tokens_for(cfg, 20, 1)
    want = zo.forward(toks, bb.as_float(W), cfg)[0]
    with block_device.Device(lva, zb.upload(ctx, cfg, W, lva.LV_F32), 512) as d:
        assert rel(d.run(toks, (1,)), want) < 2e-4


# an output row a wave, two together (from 8192 rows on; an odd number leaves half a task), and residuals of up to 2, 4 and 8 streams
@pytest.mark.parametrize("streams,width,vocab,f32", [(0, 320, 1003, False), (0, 320, 1003, True), (0, 96, 32001, False), (2, 72, 1003, False),
                                                     (3, 44, 32001, False), (5, 44, 1003, False), (5, 44, 32001, False)])
def test_logits_of_steps_read_or_not(lva, ctx, streams, width, vocab, f32):
    """a step behind one whose logits were read sends its own to the host from the output product: the same bits whatever was read before,
    for one token, several one by one and a batch, with and without all rows' logits kept, and as the greedy pick"""
    compute = lva.LV_F32 if f32 else lva.LV_BF16
    if streams:
        cfg = zb.config(width=width, vocab=vocab, streams=streams)
        model = zb.upload(ctx, cfg, zb.weights(cfg, seed=5), compute)
    else:
        cfg = bb.config(width=width, vocab=vocab, layers=[bb.layer(experts=5, top=2, ff=72)])
        model = bb.upload(ctx, cfg, bb.weights(cfg, seed=5), compute)
    a, b = lva.Session(model, 128), lva.Session(model, 128)
    toks = tokens_for(cfg, 80, 2)
    pos = 0
    for i, n in enumerate((1, 1, 1, 3, 1, 20, 1, 17, 2, 1, 18, 1, 1)):
        a.begin(toks[pos:pos + n], pos)
        want = a.logits()                                # every step
        kept = i in (4, 6, 11)                           # behind a step that was read and behind one that was not
        b.keep_all_logits(kept)
        b.begin(toks[pos:pos + n], pos)
        if kept:
            assert n == 1 and np.array_equal(b.logits_rows(0, 1)[0].view(np.uint32), want.view(np.uint32)), i
        if i % 3 == 0:
            b.wait()
        else:
            assert np.array_equal(b.logits().view(np.uint32), want.view(np.uint32)), i
            assert np.array_equal(b.logits().view(np.uint32), want.view(np.uint32)), i
        assert b.argmax() == int(want.argmax()) == a.argmax(), i
        pos += n
    a.close(); b.close(); model.close()


def test_reading_some_steps_makes_no_second_graph(lva, ctx):
    """us of the steps at which a session starts and stops to read logits, beside those of a session that always reads: the fastest of nine
    sessions.  A token's graph is made at the first of them; a second one took as long as two of these steps"""
    cfg = bb.config(width=320, vocab=1003, layers=[bb.layer(experts=5, top=2, ff=72) for _ in range(3)])
    model = bb.upload(ctx, cfg, bb.weights(cfg, seed=6), lva.LV_BF16)
    toks = tokens_for(cfg, 24, 1)

    def steps(read):
        s = lva.Session(model, 128)
        s.begin(toks[:4], 0)
        s.logits()
        out = []
        for i in range(4, len(toks)):
            t = time.perf_counter()
            s.begin(toks[i:i + 1], i)
            s.logits() if read(i) else s.argmax()
            out.append(time.perf_counter() - t)
        s.close()
        return out[1:]                                   # behind the one that makes the graph

    def fastest(read):
        return np.min([steps(read) for _ in range(9)], axis=0)

    always = np.median(fastest(lambda i: True))
    for read in (lambda i: i % 2 == 0, lambda i: i >= 12, lambda i: i < 12, lambda i: False):
        assert fastest(read).max() < 1.5 * always, (fastest(read) * 1e6, always * 1e6)
    model.close()
