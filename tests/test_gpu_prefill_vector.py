"""GPU parity against the fp64 oracle of the chunked prefill's configurations
next to the 16-bit kernel's 1, 2 and 4 query heads per kv head:

* f32 queries over f32 caches and over fp8 caches with scales, the Metal
  prefill's `float` and `float, uint8_t` instances
  (prefill_paged_attn.metal:1606, 1610; F32 dispatch at
  vasr-paged-attn/src/metal/kernels/mod.rs:119-137), on the f32 matrix
  instructions, and on the vector ALUs for at most 32 rows over 32 keys: rel
  1e-5, causal (flash varlen, eps 0) and not (the Metal kernel's 1e-6 and a
  large eps), every head dim and block size, ragged lengths, absent blocks;
* other numbers of query heads per kv head (3, 8, 16; the Metal dispatch
  takes any, mod.rs:145-283), 16-bit and fp8, on the 16-bit MFMA kernel;
* 16-bit and fp8 head-dim / block-size pairs without whole 1 KiB DMAs, on the
  vector ALUs."""

import numpy as np
import pytest
import torch

import vpa
from oracle import oracle as orc
from tests._util import (assert_attention_close, block_tables_for, make_cache, random_words,
                         to_dev, to_host, u32)

pytestmark = pytest.mark.gpu


def f8_dev(a, device):
    return torch.from_numpy(a).to(device).view(torch.float8_e4m3fn)


def vector_case(device, code, h, kvh, d, bs, prior, qlens, seed, causal=True, eps=None, fp8=False,
                scales=(1.0, 1.0), mutate_bt=None, scale=None):
    rng = np.random.default_rng(seed)
    prior = np.asarray(prior, dtype=np.int64)
    qlens = np.asarray(qlens, dtype=np.int64)
    lens = prior + qlens
    nb = int(sum((int(L) + bs - 1) // bs for L in lens)) + 8
    if fp8:
        kc = orc.fp8_from_f32((rng.standard_normal((nb, kvh, d // 16, bs, 16)) * 2)
                              .astype(np.float32))
        vc = orc.fp8_from_f32((rng.standard_normal((nb, kvh, d, bs)) * 2).astype(np.float32))
        kc_d, vc_d = f8_dev(kc, device), f8_dev(vc, device)
        ks = torch.tensor([scales[0]], dtype=torch.float32, device=device)
        vs = torch.tensor([scales[1]], dtype=torch.float32, device=device)
    else:
        kc, vc = make_cache(rng, nb, kvh, d, bs, code)
        kc_d, vc_d = to_dev(kc, code, device), to_dev(vc, code, device)
        ks = vs = None
    bt = block_tables_for(rng, [max(int(L), 1) for L in lens], nb, bs)
    if mutate_bt is not None:
        mutate_bt(bt)
    q = random_words(rng, (int(qlens.sum()), h, d), code)
    cu = np.concatenate([[0], np.cumsum(qlens)]).astype(np.uint32)
    lens32 = lens.astype(np.uint32)
    scale = d ** -0.5 if scale is None else scale
    eps = (0.0 if causal else 1e-6) if eps is None else eps
    out = vpa.paged_attention_varlen_prefill(
        to_dev(q, code, device), kc_d, vc_d, u32(bt, device), u32(lens32, device),
        u32(cu, device), ks, vs, scale, 1.0, causal=causal, denom_eps=eps)
    torch.cuda.synchronize()
    want = orc.prefill_attention(q, kc, vc, bt, lens32, cu, scale, causal=causal, dtype=code,
                                 eps=eps, kv_dtype=orc.FP8 if fp8 else None,
                                 k_scale=scales[0], v_scale=scales[1])
    return orc.to_f32(to_host(out), code), want


PRIOR = [0, 5, 31, 100, 0, 333, 16]
NEW = [1, 31, 32, 33, 129, 70, 3]


@pytest.mark.parametrize("d", [64, 96, 128, 192, 256])
@pytest.mark.parametrize("bs", [8, 16, 32])
@pytest.mark.parametrize("causal,eps", [(True, 0.0), (False, 1e-6), (True, 1e-6), (False, 0.0)])
def test_prefill_f32(device, d, bs, causal, eps):
    got, want = vector_case(device, orc.F32, 16, 8, d, bs, PRIOR, NEW,
                            seed=d + bs + 2 * causal + int(eps > 0), causal=causal, eps=eps)
    assert_attention_close(got, want, orc.F32, f"f32 d={d} bs={bs} causal={causal} eps={eps}")


@pytest.mark.parametrize("d,bs", [(128, 16), (128, 8), (64, 32), (256, 16), (96, 32)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("scales", [(1.0, 1.0), (0.37, 2.5)])
def test_prefill_f32_query_fp8_cache(device, d, bs, causal, scales):
    got, want = vector_case(device, orc.F32, 16, 8, d, bs, PRIOR, NEW, seed=d + bs + causal,
                            causal=causal, fp8=True, scales=scales)
    assert_attention_close(got, want, orc.F32, f"f32/fp8 d={d} bs={bs} causal={causal}")


@pytest.mark.parametrize("h,kvh", [(24, 8), (64, 8), (16, 1), (32, 2), (8, 8)])
@pytest.mark.parametrize("code", [orc.F32, orc.BF16, orc.F16])
def test_prefill_query_heads_per_kv_head(device, h, kvh, code):
    """3, 8 and 16 query heads per kv head (and 1), f32 on the f32 matrix
    instructions and 16-bit on the 16-bit MFMA kernel."""
    got, want = vector_case(device, code, h, kvh, 128, 16, [7, 0, 260], [40, 65, 17],
                            seed=h + kvh + code)
    assert_attention_close(got, want, code, f"h={h} kvh={kvh} code={code}")


@pytest.mark.parametrize("code,d,bs,fp8", [(orc.BF16, 96, 8, False), (orc.F16, 96, 8, False),
                                           (orc.BF16, 96, 16, True), (orc.F16, 64, 8, True),
                                           (orc.BF16, 192, 8, True)])
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_vector_16bit_shapes(device, code, d, bs, fp8, causal):
    """Head-dim / block-size pairs whose (block, head) tile is not a whole
    number of 1 KiB DMAs (no MFMA instance) on the vector kernel."""
    got, want = vector_case(device, code, 16, 8, d, bs, PRIOR, NEW, seed=d + bs + fp8 + causal,
                            causal=causal, fp8=fp8, scales=(0.8, 1.3) if fp8 else (1.0, 1.0))
    assert_attention_close(got, want, code, f"code={code} d={d} bs={bs} fp8={fp8}")


def test_prefill_f32_absent_blocks_and_large_scales(device):
    """Table entries outside the pool are skipped (their keys do not count);
    logit scales of 3 and 10 times 1/sqrt(d) (normwise at 10x, where single
    elements near zero sit at the f32 rounding of logits of size ~40)."""
    def corrupt(bt):
        bt[1, 0] = 1 << 30
        bt[3, 2] = 0xffffffff

    got, want = vector_case(device, orc.F32, 16, 8, 128, 16, PRIOR, NEW, seed=5,
                            mutate_bt=corrupt)
    assert_attention_close(got, want, orc.F32, "absent blocks")
    for factor in (3.0, 10.0):
        got, want = vector_case(device, orc.F32, 16, 8, 128, 16, PRIOR, NEW, seed=6,
                                scale=factor * 128 ** -0.5)
        num = np.sqrt(((got - want) ** 2).sum(axis=-1))
        den = np.sqrt((want ** 2).sum(axis=-1))
        assert np.max(num / np.maximum(den, 1e-300)) <= 1e-5, f"scale x{factor}"


def test_prefill_f32_row_without_keys_and_empty_sequences(device):
    """Non-causal rows of a sequence whose every block is absent see no key:
    zeros; sequences without new tokens write nothing."""
    def absent(bt):
        bt[2, :] = 1 << 30

    got, want = vector_case(device, orc.F32, 16, 8, 64, 8, [10, 0, 40, 3], [5, 0, 7, 9], seed=8,
                            causal=False, mutate_bt=absent)
    assert_attention_close(got, want, orc.F32, "no keys")
    assert not np.any(got[5:12])


@pytest.mark.parametrize("code", [orc.BF16, orc.F16])
@pytest.mark.parametrize("group,kvh,d,bs,fp8", [(3, 8, 128, 16, False), (5, 1, 64, 32, False),
                                                (7, 2, 192, 8, False), (48, 1, 96, 16, False),
                                                (130, 1, 64, 16, True), (8, 2, 256, 32, True)])
def test_prefill_any_group_keeps_f32_probabilities(device, code, group, kvh, d, bs, fp8):
    """16-bit queries with any number of query heads per kv head on the MFMA
    kernel: (position, head) row tiles of 128 rows that end inside a position
    (groups that divide neither 32 nor 128, and one above 128), 1 to 129 new
    tokens. The probabilities keep their f32 bits: next to the output's own
    rounding (half a unit in the last place, at most 2^-8 of the value in bf16
    and 2^-11 in f16) an element may be off by 2^-20, which covers f16's 22
    bits and the f32 sums, times the largest |value| behind it (below 12 here:
    6 standard deviations times the fp8 data's 2)."""
    got, want = vector_case(device, code, group * kvh, kvh, d, bs, [0, 37, 300, 1], [1, 43, 129, 2],
                            seed=group + d, causal=True, fp8=fp8)
    half = 2.0 ** -8 if code == orc.BF16 else 2.0 ** -11
    err = np.abs(got.astype(np.float64) - want)
    bound = half * np.abs(want) + 12 * 2.0 ** -20
    assert np.all(np.isfinite(got))
    assert np.max(err / bound) <= 1.0, f"worst {np.max(err / bound):.2f} of the bound"


@pytest.mark.parametrize("code", [orc.BF16, orc.F16])
@pytest.mark.parametrize("group,kvh,d,bs", [(3, 2, 128, 16), (8, 1, 64, 32), (5, 2, 256, 16)])
@pytest.mark.parametrize("n", [40, 600])
def test_prefill_any_group_cancelling_values(device, code, group, kvh, d, bs, n):
    """Values of +1 and -1 under nearly equal probabilities: the output is
    their difference, about 2^-13 of a probability, and shows every bit they
    are held in. Next to the output's own rounding an element may be off by
    2^-21: the exponent's rounding (at most 2^-22 of it at f16's offset of 7,
    times ln 2), the exponential's unit in the last place, f16's two parts
    (2^-23) and the f32 sums."""
    h, nq = group * kvh, 9
    nb = n // bs + 3
    rng = np.random.default_rng(n + d)
    kc = np.zeros((nb, kvh, d // 8, bs, 8), np.float32)
    vc = np.zeros((nb, kvh, d, bs), np.float32)
    bt = block_tables_for(rng, [n], nb, bs)
    pos = np.arange(n)
    blk, off = bt[0, pos // bs], pos % bs
    plus = (pos % 2 == 0).astype(np.float32)
    kc[blk, :, 0, off, 0] = (plus * 2.0 ** -12)[:, None]
    vc[blk, :, :, off] = (2 * plus - 1)[:, None, None]
    q = np.zeros((nq, h, d), np.float32)
    q[:, :, 0] = 1 + rng.integers(0, 64, (nq, h)) / 64  # exact in both types
    kc, vc, qw = (orc.from_f32(x, code) for x in (kc, vc, q))
    out = vpa.paged_attention_varlen_prefill(
        to_dev(qw, code, device), to_dev(kc, code, device), to_dev(vc, code, device),
        u32(bt, device), u32([n], device), u32([0, nq], device), None, None, 1.0, 1.0,
        causal=False, denom_eps=0.0)
    got = orc.to_f32(to_host(out), code).astype(np.float64)
    want = np.broadcast_to(np.tanh(q[:, :, :1].astype(np.float64) * 2.0 ** -13), got.shape)
    half = 2.0 ** -8 if code == orc.BF16 else 2.0 ** -11
    err = np.abs(got - want) / (half * np.abs(want) + 2.0 ** -21)
    assert np.max(err) <= 1.0, f"worst {np.max(err):.2f} of the bound"


@pytest.mark.parametrize("code", [orc.BF16, orc.F16])
def test_prefill_any_group_infinite_values_and_zero_scale(device, code):
    """An infinite cached value gives an infinite output (not NaN) in the rows
    that see it, and a softmax scale of 0 the mean of the visible values."""
    h, kvh, d, bs, n = 6, 2, 64, 16, 40
    rng = np.random.default_rng(3)
    kc, vc = make_cache(rng, 4, kvh, d, bs, code)
    vc = orc.to_f32(vc, code).astype(np.float32)
    vc[1, 1, 5, 3] = np.inf  # head 1, dim 5, token 3
    vc = orc.from_f32(vc, code)
    bt = np.array([[1, 2, 3]], dtype=np.uint32)
    q = random_words(rng, (n, h, d), code)
    args = (to_dev(q, code, device), to_dev(kc, code, device), to_dev(vc, code, device),
            u32(bt, device), u32([n], device), u32([0, n], device), None, None)
    out = vpa.paged_attention_varlen_prefill(*args, d ** -0.5, 1.0, causal=False)
    got = orc.to_f32(to_host(out), code)
    assert np.all(np.isposinf(got[:, 3:, 5]))
    got[:, 3:, 5] = 0
    assert np.all(np.isfinite(got))
    out = vpa.paged_attention_varlen_prefill(*args, 0.0, 1.0, causal=True)
    got = orc.to_f32(to_host(out), code)[:, :3]
    v = orc.to_f32(vc, code)[1:, 0].transpose(0, 2, 1).reshape(-1, d)[:n]
    want = np.cumsum(v.astype(np.float64), axis=0) / np.arange(1, n + 1)[:, None]
    assert_attention_close(got, np.repeat(want[:, None], 3, axis=1), code, "scale 0")


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("d,bs,n,prior", [(128, 16, 41, 70), (64, 32, 33, 5), (96, 8, 64, 129),
                                          (192, 32, 40, 40), (256, 16, 34, 30)])
def test_prefill_f32_many_short_rows(device, d, bs, n, prior, fp8):
    """Many row tiles over at most 320 keys, each sequence with more than 32
    rows: a wave of the f32 kernel takes a row tile of its own instead of a
    quarter of one tile's keys (the other cases here have fewer than 1024
    tiles, and split)."""
    if fp8 and bs == 8:
        bs = 16
    b = 129
    rng = np.random.default_rng(n)
    new = rng.integers(1, n + 1, b)
    new[0] = n
    got, want = vector_case(device, orc.F32, 8, 8, d, bs, rng.integers(0, prior + 1, b), new,
                            seed=d + n, fp8=fp8)
    assert_attention_close(got, want, orc.F32, f"d={d} bs={bs} fp8={fp8}")


@pytest.mark.parametrize("h,kvh,n", [(24, 8, 20), (16, 8, 17), (33, 11, 64)])
@pytest.mark.parametrize("causal,fp8", [(True, False), (False, False), (False, True)])
def test_prefill_f32_many_short_rows_groups(device, h, kvh, n, causal, fp8):
    """The same form with 2 and 3 query heads per kv head (row tiles that end
    inside a position), without the causal mask, and with absent blocks. (The
    fp8 codes have a standard deviation of 2; scales of 0.5 give scores and
    values the unit deviation of the f32 cases. At 1 a score of deviation 2
    alone rounds by about 2^-22, which times the largest value, 8, passes the
    floor of the bound, 1e-5 * 0.03 * 8, at one of 20 million elements.)"""
    b = 130
    rng = np.random.default_rng(n + h)
    prior, new = rng.integers(0, 90, b), rng.integers(1, n + 1, b)
    prior[0], new[0] = 60, n

    def absent(bt):
        bt[0, 1] = 0xffffffff
        bt[3, 0] = 1 << 30

    got, want = vector_case(device, orc.F32, h, kvh, 128, 16, prior, new, seed=n, causal=causal,
                            fp8=fp8, scales=(0.5, 0.5) if fp8 else (1.0, 1.0), mutate_bt=absent)
    assert_attention_close(got, want, orc.F32, f"{h} over {kvh} causal={causal} fp8={fp8}")


@pytest.mark.parametrize("d,bs", [(64, 16), (96, 32), (128, 8), (192, 16), (256, 32)])
@pytest.mark.parametrize("h,kvh,n,keys", [(8, 8, 32, 32), (8, 8, 33, 33), (8, 8, 32, 33),
                                          (16, 8, 16, 32), (16, 8, 17, 32), (24, 8, 1, 32),
                                          (24, 8, 11, 31), (16, 8, 1, 1)])
@pytest.mark.parametrize("fp8", [False, True])
def test_prefill_f32_one_tile(device, d, bs, h, kvh, n, keys, fp8):
    """Both sides of the line to the vector kernel: at most 32 rows over at
    most 32 keys."""
    if fp8 and bs == 8:
        bs = 16

    def absent(bt):
        if bt.shape[1] > 1:
            bt[0, 1] = 0xffffffff

    got, want = vector_case(device, orc.F32, h, kvh, d, bs, [keys - n, 0, max(0, keys - n - 5)],
                            [n, n, max(1, n - 1)], seed=d + n + keys, fp8=fp8, mutate_bt=absent)
    assert_attention_close(got, want, orc.F32, f"d={d} n={n} keys={keys}")
