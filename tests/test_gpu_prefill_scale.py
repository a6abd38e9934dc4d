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
    # one sequence of many keys, a short one, one without a key
    check_nan_scale(device, code, fp8, h, kvh, d, bs, [300, 7, 0], [40, 7, 2])


@pytest.mark.parametrize("code", [orc.BF16, orc.F16, orc.F32])
@pytest.mark.parametrize("h,kvh,d,bs", [(16, 8, 128, 16), (6, 2, 64, 32)])
def test_nan_scale_over_few_keys(device, code, h, kvh, d, bs):
    """At most 32 keys: f32 queries on the vector kernel."""
    for fp8 in (False, True):
        check_nan_scale(device, code, fp8, h, kvh, d, bs, [32, 7, 0], [5, 7, 2])


@pytest.mark.parametrize("code,fp8,d,bs", [(orc.BF16, False, 96, 8), (orc.F16, False, 96, 8),
                                           (orc.BF16, True, 64, 8), (orc.F16, True, 96, 16)])
def test_nan_scale_without_whole_tiles(device, code, fp8, d, bs):
    """The 16-bit queries' shapes on the vector kernel, over several tiles."""
    check_nan_scale(device, code, fp8, 8, 4, d, bs, [70, 7, 0], [9, 7, 2])


def check_nan_scale(device, code, fp8, h, kvh, d, bs, lens, new):
    rng = np.random.default_rng(d + h)
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
            rows = sum(new) - new[-1]  # the last sequence has no key
            assert np.all(np.isnan(got[:rows])), f"scale {scale} causal={causal}"
            assert not np.any(got[rows:])
