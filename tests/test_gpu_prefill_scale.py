"""GPU chunked prefill with a softmax scale that is not a number: a NaN
``softmax_scale``, or a NaN ``k_scale`` (device data no host check sees), makes
every row that sees a key NaN in each of the prefill kernels, as the decode
does over the same cache, and leaves rows without a key at zero."""

import numpy as np
import pytest
import torch

import vpa
from oracle import oracle as orc
from tests._util import block_tables_for, make_cache, random_words, to_dev, to_host, u32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("code", [orc.BF16, orc.F16, orc.F32])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("h,kvh,d,bs", [(8, 8, 128, 16), (16, 8, 128, 16), (16, 4, 64, 32),
                                        (12, 4, 128, 32), (8, 4, 192, 16)])
def test_nan_scale_gives_nan(device, code, fp8, h, kvh, d, bs):
    rng = np.random.default_rng(d + h)
    # one sequence of many keys, a short one, one without a key
    lens, new = [300, 7, 0], [40, 7, 2]
    nb = 48
    if fp8:
        x = 16
        kc, vc = ((torch.randn(s, device=device) * 2).to(torch.float8_e4m3fn)
                  for s in ((nb, kvh, d // x, bs, x), (nb, kvh, d, bs)))
    else:
        kc, vc = (to_dev(w, code, device) for w in make_cache(rng, nb, kvh, d, bs, code))
    bt = block_tables_for(rng, [max(n, 1) for n in lens], nb, bs)
    q = random_words(rng, (sum(new), h, d), code)
    cu = np.concatenate([[0], np.cumsum(new)])
    one = torch.ones(1, device=device) if fp8 else None
    nan = torch.full((1,), float("nan"), device=device)
    cases = [(float("nan"), one)] + ([(d ** -0.5, nan)] if fp8 else [])
    for scale, k_scale in cases:
        for causal in (True, False):
            out = vpa.paged_attention_varlen_prefill(
                to_dev(q, code, device), kc, vc, u32(bt, device), u32(lens, device),
                u32(cu, device), k_scale, one, scale, 1.0, causal=causal)
            torch.cuda.synchronize()
            got = orc.to_f32(to_host(out), code)
            assert np.all(np.isnan(got[:47])), f"scale {scale} causal={causal}"
            assert not np.any(got[47:])
