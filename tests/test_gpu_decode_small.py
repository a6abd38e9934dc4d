"""GPU parity of the decode's small-grid form (at most 64 sequences: no work
list, chunk length worked out on the device) and of the work list's two chunk
lengths, against the fp64 oracle, at the sizes where each takes over: one
chunk up to a maximum of 512 tokens; chunks of 256, 512 and 1024 tokens up to
128 (sequence, kv head) pairs; above, the list, with 2048-token chunks, or
1024-token ones where the maximum exceeds 2048 and there are at most 512
pairs. Lengths sit on both sides of tiles and chunks,
with empty contexts, absent blocks and a maximum (as frozen in a captured
graph) above every length. The list's cases have enough sequences for it at
every number of kv heads here."""

import numpy as np
import pytest
import torch

import vpa
from oracle import oracle as orc
from tests._util import (assert_attention_close, block_tables_for, make_cache, random_words,
                         to_dev, to_host, u32)

pytestmark = pytest.mark.gpu

CASES = {
    "one_chunk": ([512, 1, 16, 17, 0, 497, 496, 129], 512),
    "one_chunk_64": ([(37 * i) % 513 for i in range(64)], 512),
    "one_sequence": ([1], 1),
    "chunk_256": ([513], 513),
    "chunk_256_frozen": ([0, 255, 256, 257, 1, 1023], 4096),
    "chunk_256_two": ([3000, 2049], 3000),
    "chunk_512": ([1500, 1024, 1537, 1, 0, 1536, 1025, 1999], 2048),
    "chunk_1024": ([3000 + 7 * i for i in range(14)] + [1024, 1025], 4096),
    "list_1024": ([600 + 91 * i for i in range(16)] + [1024, 2048, 0] + [90] * 21, 2200),
    "list_one_chunk": ([130 + 5 * i for i in range(40)], 1024),
    "list_2048": ([(53 * i) % 700 for i in range(64)] + [2048, 2049], 2049),
    "list_1024_full": ([1100 + 37 * i for i in range(24)] + [1024, 1] + [300] * 8, 4096),
}


def setup(device, code, h, kvh, d, bs, lens, max_ctx, seed, absent=True):
    rng = np.random.default_rng(seed)
    nb = sum((int(n) + bs - 1) // bs for n in lens) + 8
    kc, vc = make_cache(rng, nb, kvh, d, bs, code)
    bt = block_tables_for(rng, [max(int(n), 1) for n in lens], nb, bs)
    cols = (max_ctx + bs - 1) // bs
    bt = np.pad(bt, ((0, 0), (0, max(0, cols - bt.shape[1]))))
    if absent and len(lens) > 1 and lens[0] > bs:
        bt[0, 0] = 0xffffffff  # a block outside the pool: its tokens are skipped
    q = random_words(rng, (len(lens), h, d), code)
    lens = np.asarray(lens, dtype=np.uint32)
    return q, kc, vc, bt, lens


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("code,h,kvh,d,bs", [(orc.BF16, 16, 8, 128, 16), (orc.F16, 16, 4, 64, 32),
                                             (orc.BF16, 8, 8, 192, 8), (orc.BF16, 16, 8, 128, 32)])
def test_decode_small_grid_and_list(device, name, code, h, kvh, d, bs):
    lens, max_ctx = CASES[name]
    q, kc, vc, bt, lens = setup(device, code, h, kvh, d, bs, lens, max_ctx, seed=len(lens) + d)
    args = (to_dev(q, code, device), None, None, to_dev(kc, code, device),
            to_dev(vc, code, device), u32(bt, device), u32(lens, device), None, max_ctx,
            d ** -0.5, 1.0, None)
    ws = vpa.paged_attention_workspace(len(lens), h, d, max_ctx, device)
    ws.fill_(0xff)  # NaN partial rows, were any read that was not written
    out = vpa.paged_attention(*args, workspace=ws)
    ws.fill_(0xff)
    vpa.paged_attention_plan(args[6], max_ctx, bt.shape[1], h, args[3], args[4], args[0].dtype, ws)
    planned = vpa.paged_attention(*args, workspace=ws, planned=True)
    torch.cuda.synchronize()
    want = orc.paged_attention(q, kc, vc, bt, lens, max_ctx, d ** -0.5, dtype=code)
    got = orc.to_f32(to_host(out), code)
    assert_attention_close(got, want, code, name)
    assert not np.any(got[lens == 0])
    assert torch.equal(out.view(torch.int16), planned.view(torch.int16))


@pytest.mark.parametrize("name", ["one_chunk", "one_sequence", "chunk_256", "chunk_512",
                                  "chunk_1024", "list_1024"])
@pytest.mark.parametrize("h,kvh,d,bs", [(16, 8, 128, 16), (8, 8, 128, 32), (16, 4, 96, 32)])
def test_decode_small_grid_append(device, name, h, kvh, d, bs):
    """The append fused into the small-grid form against the two calls, bit
    for bit: outputs and cache bytes."""
    lens, max_ctx = CASES[name]
    lens = [max(n, 1) for n in lens]
    code = orc.BF16
    q, kc, vc, bt, lens = setup(device, code, h, kvh, d, bs, lens, max_ctx, seed=d + h,
                                absent=False)
    rng = np.random.default_rng(9)
    k, v = (to_dev(random_words(rng, (len(lens), kvh, d), code), code, device) for _ in "kv")
    pos = lens.astype(np.int64) - 1
    slots = bt[np.arange(len(lens)), pos // bs].astype(np.int64) * bs + pos % bs
    q_d, bt_d, len_d = to_dev(q, code, device), u32(bt, device), u32(lens, device)
    a = [to_dev(kc, code, device), to_dev(vc, code, device)]
    b = [x.clone() for x in a]
    vpa.reshape_and_cache(k, v, None, None, *a, torch.from_numpy(slots).to(device))
    two = vpa.paged_attention(q_d, None, None, *a, bt_d, len_d, None, max_ctx, d ** -0.5, 1.0, None)
    one = vpa.reshape_and_cache_paged_attention(q_d, k, v, None, None, *b, bt_d, len_d, max_ctx,
                                                d ** -0.5)
    torch.cuda.synchronize()
    for x, y in zip([two] + a, [one] + b):
        assert torch.equal(x.view(torch.int16), y.view(torch.int16))


@pytest.mark.parametrize("seqs,kvh,lo,hi,max_ctx", [
    (24, 8, 1228, 2048, 4096), (64, 8, 400, 2049, 2049),
    (24, 8, 1228, 2048, 2048),  # one chunk reaches the maximum
    (65, 8, 1, 4096, 4096),     # more than 512 pairs
    (200, 1, 900, 3000, 3000)])
def test_list_chunk_length(device, seqs, kvh, lo, hi, max_ctx):
    """The list's header: log2 of its chunk length and the number of items
    (1024-token chunks above 2048 tokens for up to 512 pairs, else 2048), and
    the decode over it against the oracle."""
    h, d, bs = 2 * kvh, 64, 16
    rng = np.random.default_rng(seqs + hi)
    lens = rng.integers(lo, hi, size=seqs, endpoint=True)
    lens[:2] = lo, hi
    q, kc, vc, bt, lens = setup(device, orc.BF16, h, kvh, d, bs, [int(x) for x in lens], max_ctx,
                                seed=seqs)
    args = (to_dev(q, orc.BF16, device), None, None, to_dev(kc, orc.BF16, device),
            to_dev(vc, orc.BF16, device), u32(bt, device), u32(lens, device), None, max_ctx,
            d ** -0.5, 1.0, None)
    ws = vpa.paged_attention_workspace(seqs, h, d, max_ctx, device)
    ws.fill_(0xff)
    vpa.paged_attention_plan(args[6], max_ctx, bt.shape[1], h, args[3], args[4], torch.bfloat16, ws)
    header = ws[-256:].view(torch.int32)[:2].tolist()
    chunk = 1024 if max_ctx > 2048 and seqs * kvh <= 512 else 2048
    assert header == [chunk.bit_length() - 1,
                      int(np.sum((lens.astype(np.int64) + chunk - 1) // chunk))]
    out = vpa.paged_attention(*args, workspace=ws, planned=True)
    torch.cuda.synchronize()
    want = orc.paged_attention(q, kc, vc, bt, lens, max_ctx, d ** -0.5, dtype=orc.BF16)
    assert_attention_close(orc.to_f32(to_host(out), orc.BF16), want, orc.BF16)


@pytest.mark.parametrize("b,max_ctx,parts", [(1, 1, 0), (1, 129, 0), (3, 200, 0), (2, 256, 0),
                                             (2, 257, 3), (1, 512, 4), (40, 512, 2)])
def test_f32_partitions(device, b, max_ctx, parts):
    """f32 decode: up to one whole partition (256 tokens) a call writes its
    output alone (no partial rows, so no second launch to merge them); above,
    half partitions where whole ones leave SIMDs idle, whole ones else.
    parts: the partial rows of a sequence and head."""
    h, kvh, d, bs = 16, 8, 64, 16
    lens = [max_ctx] * b
    q, kc, vc, bt, lens = setup(device, orc.F32, h, kvh, d, bs, lens, max_ctx, seed=b + max_ctx,
                                absent=False)
    ws = vpa.paged_attention_workspace(b, h, d, max_ctx, device)
    ws.fill_(0xff)
    out = vpa.paged_attention(
        to_dev(q, orc.F32, device), None, None, to_dev(kc, orc.F32, device),
        to_dev(vc, orc.F32, device), u32(bt, device), u32(lens, device), None, max_ctx, d ** -0.5,
        1.0, None, workspace=ws)
    torch.cuda.synchronize()
    want = orc.paged_attention(q, kc, vc, bt, lens, max_ctx, d ** -0.5, dtype=orc.F32)
    assert_attention_close(to_host(out), want, orc.F32, f"f32 {b} x {max_ctx}")
    written = int((ws.view(torch.int32) != -1).sum())
    assert (written > 0) == (parts > 0)
    # each partial row is head_dim outputs, a maximum and a sum
    assert abs(written - b * h * parts * (d + 2)) <= written // 100
