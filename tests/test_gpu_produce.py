"""The producer's workgroup layouts: a slot per wave on an idle card, several per
wave, every slot of a token; elements per lane from one to eight; with and without
norms.  Every layout does the same arithmetic, so one call over many tokens equals
the calls over its parts bit for bit, and the rows equal the oracle's rmsnorm and
rotary within two ulps of the rotation's larger operand: each operand may be an ulp
off where the FP64 norm sits at a rounding tie, and |cos| and |sin| are at most 1."""

import numpy as np
import pytest

from gpu_util import host, log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("hq,hkv,D,tokens", [(2, 1, 6, 1100), (14, 2, 64, 1030), (5, 5, 96, 70), (16, 8, 128, 1025),
                                             (32, 8, 128, 65), (8, 4, 256, 1024), (4, 1, 320, 40), (3, 1, 512, 300)])
def test_producer_layouts(orc, hq, hkv, D, tokens, norm):
    import torch

    from toklet_amd import ops

    rng = np.random.default_rng(D + tokens)
    ctx = ops.Context(0)
    x = [rng.standard_normal((tokens, h, D)).astype(np.float32) for h in (hq, hkv, hkv)]
    w = (1 + 0.1 * rng.standard_normal(D)).astype(np.float32)
    xd = [torch.from_numpy(a).cuda() for a in x]
    wd = torch.from_numpy(w).cuda() if norm else None

    def call(a, b):
        q = torch.full((b - a, hq, D), np.nan, device="cuda")
        k, v = (torch.full((hkv, b - a, D), np.nan, device="cuda") for _ in range(2))
        ops.produce_qkv(ctx, ops.ProducerShape(b - a, hq, hkv, D, 50 + a, theta=1e6), *(t[a:b] for t in xd), wd, wd, q, k, v,
                        (b - a) * D)
        return host(q), host(k).transpose(1, 0, 2), host(v).transpose(1, 0, 2)

    whole = call(0, tokens)
    cuts = [0, 1, 20, tokens]
    parts = [np.concatenate(p) for p in zip(*(call(a, b) for a, b in zip(cuts, cuts[1:])))]
    for a, b in zip(whole, parts):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
    for got, a, h in ((whole[0], x[0], hq), (whole[1], x[1], hkv)):
        y = orc.rmsnorm(a.reshape(-1), w, tokens * h, D, 1e-6) if norm else a.reshape(-1)
        ref = np.asarray(orc.rotary(y, tokens, h, D, 50, 1e6), np.float32).reshape(got.shape)
        worst = np.max(np.abs(got - ref) / np.spacing(np.maximum(np.abs(ref), np.abs(y.reshape(got.shape)))))
        log(f"{hq}/{hkv}/{D} x {tokens}, norm {norm}: {worst:.2f} ulp")
        assert worst <= 2
    assert np.array_equal(whole[2], x[2])
    ctx.close()
