"""tkh_logit_softcap at the sizes where it changes form: one workgroup's share, its
largest input, the first two-launch size, and a vocabulary.  Bar: FP64 tanh
rounded once to FP32, so at most one FP32 ulp from the oracle's."""

import numpy as np
import pytest

from gpu_util import host, log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 1023, 1025, 2048, 2049, 65537, 262144, 1 << 21])
def test_softcap_sizes(orc, n):
    import torch

    from toklet_amd import ops

    ctx = ops.Context(0)
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n) * 40).astype(np.float32)
    t = torch.from_numpy(x).cuda()
    ops.logit_softcap(ctx, t, 30.0)
    got, ref = host(t), np.asarray(orc.logit_softcap(x, 30.0), np.float32)
    ulp = np.max(np.abs(got.view(np.int32).astype(np.int64) - ref.view(np.int32)))
    log(f"softcap of {n}: {ulp} ulp")
    assert ulp <= 1
    # A non-finite value anywhere: the error, and nothing is written; then a
    # finite call works again.
    for at in {0, n // 2, n - 1}:
        bad = x.copy()
        bad[at] = np.inf
        t = torch.from_numpy(bad).cuda()
        with pytest.raises(ops.TkhError) as e:
            ops.logit_softcap(ctx, t, 30.0)
        assert e.value.name == "NonFinite"
        assert np.array_equal(host(t).view(np.uint32), bad.view(np.uint32))
    t = torch.from_numpy(x).cuda()
    ops.logit_softcap(ctx, t, 30.0)
    assert np.array_equal(host(t).view(np.uint32), got.view(np.uint32))
    ctx.close()
