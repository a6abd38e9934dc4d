"""GPU parity of the 16-bit MFMA prefill on both sides of its split rule (head
dim 128): few row tiles, whose workgroups split a tile's keys over their
waves, and the same sequences among enough others that they do not, against
the fp64 oracle. Key counts on both sides of a tile (32), a step of four tiles
(128) and the rule's 64 and, for at most 64 rows, 192."""

import numpy as np
import pytest

from oracle import oracle as orc
from tests._util import assert_attention_close
from tests.test_gpu_prefill_vector import vector_case

pytestmark = pytest.mark.gpu

# (prior, new) tokens; with 16 heads over 8, at most 256 tiles of 32 rows but
# for the last two
FEW = {
    "one_token": ([600], [1]),
    "keys_65": ([0], [65]),
    "keys_64": ([0, 31], [64, 33]),
    "few_rows_192": ([176, 100], [16, 3]),
    "few_rows_193": ([177, 100], [16, 3]),
    "ragged": ([0, 127, 513, 0], [128, 1, 31, 0]),
    "long": ([1000], [300]),
    "many_keys": ([511, 300], [200, 250]),
    "two_per_cu": ([511, 300], [200, 260]),  # 272 tiles: not split
    "two_per_cu_long": ([0], [528]),  # 264 tiles of one chunk: split where causal
}


@pytest.mark.parametrize("name", FEW)
@pytest.mark.parametrize("code,h,kvh,bs,fp8", [(orc.BF16, 16, 8, 16, False),
                                               (orc.F16, 8, 8, 32, False),
                                               (orc.BF16, 16, 4, 16, True),
                                               (orc.F16, 12, 4, 32, False)])
@pytest.mark.parametrize("many", [False, True])
def test_prefill_split_keys(device, name, code, h, kvh, bs, fp8, many):
    prior, new = (list(x) for x in FEW[name])
    if many:  # 40 more sequences of 1 to 40 tokens: past the rule
        prior += [5 * i % 37 for i in range(40)]
        new += [i + 1 for i in range(40)]

    def absent(bt):
        if prior[0] > 2 * bs:
            bt[0, 1] = 0xffffffff  # a block outside the pool

    for causal in (True, False):
        got, want = vector_case(device, code, h, kvh, 128, bs, prior, new, seed=len(prior) + h,
                                causal=causal, fp8=fp8, mutate_bt=absent)
        assert_attention_close(got, want, code, f"{name} causal={causal} many={many}")
        assert np.all(np.isfinite(got))


def test_prefill_split_epsilon_and_no_keys(device):
    """A large denominator epsilon (relative to the row's true maximum over
    all waves), and rows whose every block is absent: zeros."""
    def absent(bt):
        bt[1, :] = 1 << 30

    got, want = vector_case(device, orc.F16, 16, 8, 128, 16, [300, 80], [40, 20], seed=4,
                            causal=False, eps=0.7, mutate_bt=absent)
    assert_attention_close(got, want, orc.F16, "eps")
    assert not np.any(got[40:])
