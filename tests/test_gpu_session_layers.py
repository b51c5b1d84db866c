"""A session whose layers' inputs are given together (evaluate) launches several
layers at once; the contexts equal the layer-by-layer calls' bit for bit: more
layers than one launch holds, windows of different split layouts and wave counts,
shared layers behind their owners, and a layer whose Q projection is an earlier
layer's context, which has to wait for it."""

import numpy as np
import pytest

from gpu_util import TOL_HALF, host, log, max_err, stored

pytestmark = pytest.mark.gpu

# (hq, hkv, D, storage, windows, shared, softcap, feed): feed (a, b) makes layer b's
# q_proj the context buffer of layer a.
CASES = [
    (16, 8, 128, "bf16", [0] * 11, 0, 0.0, None),
    (8, 4, 256, "bf16", [40, 200, 0, 40, 200, 40, 0, 200, 40, 0], 0, 50.0, (2, 3)),
    (14, 2, 64, "f16", [0, 33, 0, 33, 0], 2, 0.0, (0, 1)),
    (8, 4, 256, "f16", [300, 100, 300, 0, 0, 300], 2, 0.0, None),
    (14, 2, 64, "f32", [0, 30, 0], 0, 0.0, None),
]


@pytest.mark.parametrize("queued", [True, False])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}-{c[3]}-{len(c[4])}")
def test_layers_together_equal_layer_by_layer(case, queued):
    import torch

    from toklet_amd import ops, session as sm

    hq, hkv, D, storage, windows, shared, softcap, feed = case
    prompt, steps, layers = 260, 5, len(windows)
    total = prompt + steps
    rng = np.random.default_rng(D + layers)
    f = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda()
    proj = [(f(total, hq, D), f(total, hkv, D), f(total, hkv, D)) for _ in windows]
    wq, wk = f(D) * 0.02 + 1, f(D) * 0.02 + 1
    ctx = ops.Context(0, synchronous=not queued)
    got = []
    for together in (True, False):
        outs = [torch.full((total, hq, D), np.nan, device="cuda") for _ in windows]
        s = sm.Session(ctx, sm.Options(capacity=total, prefill_chunk_size=100, layers=layers, query_heads=hq, kv_heads=hkv,
                                       head_dim=D, storage=storage, score_scale=1.0 / np.sqrt(D), softcap=softcap,
                                       layer_windows=windows, shared_layers=shared))
        io = [sm.LayerIo(outs[feed[0]] if feed and l == feed[1] else q, k, v, o, wq, wk)
              for l, ((q, k, v), o) in enumerate(zip(proj, outs))]
        s.set_tokens([1] * prompt)
        if together:
            s.evaluate(io)
            s.append([2] * steps)
            s.evaluate(io, chunk_limit=1)
        else:
            for limit in (100, 1):
                while True:
                    start, n = s.chunk_begin(limit)
                    if n == 0:
                        break
                    for l, x in enumerate(io):
                        s.chunk_layer(l, sm.LayerIo(*(t[start:start + n] for t in (x.q_proj, x.k_proj, x.v_proj, x.context)),
                                                    wq, wk))
                    s.chunk_commit()
                s.append([2] * (steps if limit == 100 else 0))
        s.synchronize()
        got.append([host(o) for o in outs])
        s.close()
    for l in range(layers):
        same = np.array_equal(got[0][l].view(np.uint32), got[1][l].view(np.uint32))
        log(f"{case[:4]} layer {l} of {layers}, queued {queued}: identical {same}")
        assert same and np.all(np.isfinite(got[0][l]))
    ctx.close()


# (hq, hkv, D, chunk, prompt, windows, workspace, environment): the ways a chunk's
# layers can fail to share a launch.
SEPARATE = [
    # Few tokens: the producers go out together, the attention of each layer is the
    # streaming decode kernel's.
    (16, 8, 128, 3, 50, [0, 0, 33, 0], 0, {}),
    (8, 4, 256, 2, 31, [40, 0, 12, 40], 0, {}),
    # A workspace that holds the split partials of some of the layers.
    (8, 4, 256, 100, 700, [0] * 6, 5 << 20, {}),
    (14, 2, 64, 100, 900, [0, 200, 0, 200, 0], 3 << 20, {}),
    # The 32-row kernel, of which there is no build for several layers at 128 and 256.
    (16, 8, 128, 100, 260, [0, 0, 33, 0], 0, {"TKH_PREFILL16": "0"}),
    (8, 4, 256, 100, 260, [40, 0, 200, 40], 0, {"TKH_PREFILL16": "0"}),
]


@pytest.mark.parametrize("case", SEPARATE, ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}-{c[3]}-{c[6]}-{len(c[7])}")
def test_layers_that_do_not_share_a_launch(orc, case, monkeypatch):
    import torch

    from toklet_amd import ops, session as sm

    hq, hkv, D, chunk, prompt, windows, workspace, environment = case
    for name, value in environment.items():
        monkeypatch.setenv(name, value)
    rng = np.random.default_rng(D + prompt)
    f = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda()
    proj = [(f(prompt, hq, D), f(prompt, hkv, D), f(prompt, hkv, D)) for _ in windows]
    scale = 1.0 / np.sqrt(D)
    ctx = ops.Context(0, synchronous=False, workspace_bytes=workspace)
    got = []
    for together in (True, False):
        outs = [torch.full((prompt, hq, D), np.nan, device="cuda") for _ in windows]
        s = sm.Session(ctx, sm.Options(capacity=prompt, prefill_chunk_size=chunk, layers=len(windows), query_heads=hq,
                                       kv_heads=hkv, head_dim=D, storage="bf16", score_scale=scale, theta=1e4,
                                       layer_windows=windows))
        io = [sm.LayerIo(*p, o) for p, o in zip(proj, outs)]
        s.set_tokens([1] * prompt)
        if together:
            s.evaluate(io)
        else:
            while True:
                start, n = s.chunk_begin(chunk)
                if n == 0:
                    break
                for l, x in enumerate(io):
                    s.chunk_layer(l, sm.LayerIo(*(t[start:start + n] for t in (x.q_proj, x.k_proj, x.v_proj, x.context))))
                s.chunk_commit()
        s.synchronize()
        got.append([host(o) for o in outs])
        s.close()
    ctx.close()
    for l, window in enumerate(windows):
        assert np.array_equal(got[0][l].view(np.uint32), got[1][l].view(np.uint32)), f"layer {l}"
        q, k = (stored(np.asarray(orc.rotary(host(x).reshape(-1), prompt, h, D, 0, 1e4), np.float32), "bf16")
                for x, h in zip(proj[l], (hq, hkv)))
        k = np.ascontiguousarray(k.reshape(prompt, hkv, D).transpose(1, 0, 2))
        v = np.ascontiguousarray(stored(host(proj[l][2]), "bf16").transpose(1, 0, 2))
        ref, _, _ = orc.window_attention(q, k.reshape(-1), v.reshape(-1), prompt, prompt, prompt, hq, hkv, D, 0, 0,
                                         window or None, scale)
        err = max_err(got[0][l].reshape(-1), ref)
        log(f"{case[:6]} layer {l}: max abs error {err:.2e}")
        assert err <= TOL_HALF
