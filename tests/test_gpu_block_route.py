"""The choice of experts: equal router rows tie to the last bit and the lower index wins, in one-token steps and in batches; on both
sides of 64 experts, where the choice of a token takes another form.

Small integers as embeddings, norm weights of one and router rows that come in equal pairs: an odd number of experts a token cuts a
pair.  The plain evaluation chooses by the same rule (choose_experts); a wrong pick is an error of order one."""
import numpy as np
import pytest

import block_builder as bb
import block_device
import block_oracle as bo
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
