"""The tiles and K slices of bfloat16 products of many tokens, at sizes around their edges: a feed-forward between an embedding and the
logits (mixers add nothing), dense and chosen by a router.

The tolerance is the rounding itself: what the plain evaluation moves by when its product operands are rounded to bfloat16, twice over
(roundings of 32-bit values that fall on the other side).  A tile, a slice or a row in the wrong place is an error of order one."""
import numpy as np
import pytest

import block_builder as bb
import block_oracle as bo
import zedenex_builder as zb
import zedenex_oracle as zo
from block_device import Device, rel, tokens_for

pytestmark = pytest.mark.gpu
BF16 = 30


def rounded(a):
    return bb.from_bf16(bb.to_bf16(a))


def dense_model(toks, W, cfg, r):
    x = np.stack([zo.embedding(toks, W, cfg["embedding"])] * cfg["streams"])
    x = zo.spread_streams(x, W["l0.hc1.mix"], W["l0.hc1.out"], 0 * x[0])
    h = r(zo.norm(zo.gather_streams(x, W["l0.hc2.in"]), W, "l0.norm2", cfg["norm"]["eps"]))
    a = np.maximum(h @ W["l0.mlp.gate"].T, 0) * (h @ W["l0.mlp.up"].T)
    x = zo.spread_streams(x, W["l0.hc2.mix"], W["l0.hc2.out"], r(a) @ W["l0.mlp.down"].T)
    return r(zo.norm(x.sum(0), W, "final.norm", cfg["norm"]["eps"])) @ W["embed"].T


def check_last(d, toks, want, tol):
    """the last token's logits alone: it takes in the pending slices or experts in front of the head, on another path than all rows"""
    d.sess.keep_all_logits(False)
    d.sess.begin(toks, 0)
    assert rel(d.sess.logits()[None], want[-1:]) < tol * max(1.0, np.sqrt(np.mean(want ** 2) / np.mean(want[-1] ** 2)))


# width, feed-forward, tokens.  Columns (64 a K step): 1, 3, 11 and more steps in front of the pipelines' two and three stages; rows and
# tokens one beside a tile's edge; feed-forwards whose way down is cut into 2 and 4 slices, the last one shorter
DENSE = [(40, 4100, 1100), (130, 2060, 1030), (700, 2060, 1025), (700, 4100, 1281), (300, 1100, 129), (300, 2113, 127), (257, 4160, 257),
         (1030, 3000, 255), (128, 2048, 513), (129, 1025, 65)]
# products down in 1 to 4 slices (what the plan takes of each: test_host_plans.py)
DENSE += [(1536, 2500, 700), (4100, 1100, 900), (3000, 2060, 900), (2500, 2500, 777), (1536, 3000, 900), (4100, 3000, 900), (4102, 2500, 897)]
# few columns and many rows: 128 x 128, a rest of every number of units of 32 tokens
DENSE += [(70, 5500, 641), (70, 7000, 513), (70, 8200, 385), (70, 11008, 257), (70, 8200, 449), (70, 4100, 960)]
DENSE += [(70, 10240, 961), (70, 5500, 801), (70, 7000, 641), (70, 11008, 289), (70, 11008, 321), (70, 11008, 353)]
# gate and up in 256 rows x 128, 160, 192 and 256 tokens: no rest, and rests of every number of units of 32, one token beside a unit's end
WIDE_DENSE = [(2875, 286, 129), (4418, 306, 161), (929, 8448, 193), (1143, 8440, 225), (1103, 4325, 512)]
WIDE_DENSE += [(327, 8923, 480), (323, 5868, 641), (327, 6574, 513), (325, 8533, 385), (321, 8272, 417), (367, 8343, 449)]
WIDE_DENSE += [(257, 6324, 960), (260, 4994, 961), (393, 5410, 801), (261, 6857, 641), (385, 8237, 481), (129, 8953, 1281), (277, 6360, 929)]
WIDE_DENSE += [(322, 7533, 1024), (326, 5958, 1025), (329, 8097, 801), (325, 6622, 897), (327, 6373, 1009)]
# ... of 2 and 3 K steps, as many as the stages
WIDE_DENSE += [(100, 15500, 1793), (100, 15000, 1921), (150, 16500, 1793), (150, 12500, 1921), (150, 12500, 897), (150, 10500, 1921)]
# down in one slice of 160, 192 and 256 tokens, and in slices of 128, 160 and 192 of which the last one is shorter
WIDE_DENSE += [(5995, 505, 1291), (8329, 505, 1122), (7681, 405, 1559), (7188, 1447, 257), (8815, 1760, 129), (5660, 2742, 129), (8251, 1675, 385), (7180, 4288, 257), (6524, 2700, 641)]
DENSE += WIDE_DENSE
# streams so wide that the sum of slices and the norm's input would not fit LDS side by side
DENSE += [(20544, 1152, 33)]


@pytest.mark.parametrize("width,ff,n", DENSE)
def test_dense_tiles(lva, ctx, width, ff, n):
    cfg = zb.config(width=width, streams=2, layers=[zb.layer(zb.ssm(), ff=ff)])
    W = zb.weights(cfg, seed=n)
    W["l0.mix.o"][:] = 0
    toks, F = tokens_for(cfg, n, 1), bb.as_float(W)
    want = dense_model(toks, F, cfg, lambda a: a)
    tol = 2 * rel(dense_model(toks, F, cfg, rounded), want)
    assert tol < 2e-2
    with Device(lva, zb.upload(ctx, cfg, W, BF16), 2048) as d:
        assert rel(d.run(toks, (n,)), want) < tol
        check_last(d, toks, want, tol)


def test_slices_do_not_hang_on_what_came_before(lva, ctx):
    """the same tokens give the same bits in a new session and behind a batch that has grown its workspace past 1024 tokens"""
    cfg = zb.config(width=700, streams=2, layers=[zb.layer(zb.ssm(), ff=4100)])
    W = zb.weights(cfg, seed=4)
    with Device(lva, zb.upload(ctx, cfg, W, BF16), 2048) as d:
        for n in (300, 777, 129):
            toks = tokens_for(cfg, n, 1)
            first = d.run(toks, (n,))
            d.run(tokens_for(cfg, 1100, 2), (1100,))
            assert np.array_equal(d.run(toks, (n,)), first), n


# what the plan takes of each: test_host_plans.py
EXPERTS = [(130, 1100, 900, 4, 2), (40, 2050, 513, 9, 3), (700, 700, 1281, 5, 2), (257, 130, 1030, 12, 4), (64, 24, 17, 3, 2), (130, 520, 230, 4, 2), (70, 300, 375, 3, 2)]
# gate and up, down in tiles of 256 rows, one or several an expert; an expert after the other, with either tile, one or several
EXPERTS += [(2886, 126, 52, 5, 2), (2080, 847, 539, 12, 3), (167, 2357, 43, 32, 2), (677, 2191, 1210, 24, 3), (138, 1381, 212, 130, 4), (1030, 200, 2000, 128, 9),
            (40, 24, 1900, 128, 9), (103, 94, 116, 130, 4)]


@pytest.mark.parametrize("width,ff,n,experts,top", EXPERTS)
def test_expert_tiles(lva, ctx, width, ff, n, experts, top):
    cfg = bb.config(width=width, layers=[bb.layer(experts=experts, top=top, ff=ff)])
    W = bb.weights(cfg, seed=n)
    for s in ("left", "right"):
        W[f"l0.mix.{s}.o"][:] = 0
    F, eps = bb.as_float(W), cfg["norm"]["eps"]

    def model(toks, r):
        x = F["embed"][toks]
        h = bo.rms_norm(x, F["l0.norm2"], eps)
        y = np.zeros_like(x)
        z = h @ F["l0.mlp.router"].T                      # the choice by 32-bit scores; tokens whose choice hangs on less are not asked
        for e in range(experts):
            t = np.nonzero((bo.choose_experts(z, top) == e).any(1))[0]
            a = r(bo.sigmoid(z[t, e])[:, None] * h[t])
            p = f"l0.mlp.e{e}."
            y[t] += r(bo.silu(a @ F[p + "gate"].T) * (a @ F[p + "up"].T)) @ F[p + "down"].T
        return r(bo.rms_norm(x + bo.rms_norm(y, F["l0.norm2b"], eps), F["final.norm"], eps)) @ F["head"].T, np.sort(z, 1)[:, ::-1]

    toks = tokens_for(cfg, 4 * n, 1)
    z = model(toks, lambda a: a)[1]
    toks = toks[z[:, top - 1] - z[:, top] > 0.02][:n]
    assert len(toks) == n
    want = model(toks, lambda a: a)[0]
    tol = 2 * rel(model(toks, rounded)[0], want)
    assert tol < 4e-2
    with Device(lva, bb.upload(ctx, cfg, W, BF16), 2048) as d:
        assert rel(d.run(toks, (n,)), want) < tol
        check_last(d, toks, want, tol)
