"""Attention of runs of rows over several sequences of one length, whose groups are taken by length (attn_rows.inl): lengths that fill no group and no run, sequences that go on from cached keys, more
groups of some sequences than of others, one sequence that is another length where the table's look does not or does see it, key splits.  The reference is run()'s float64 softmax and its bound:
fp32 products of up to 600 terms and exponentials at 1e-6, 1e-5 of the largest value."""
import pytest

from tests.test_gpu_attn_rows import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spans,H,G,d,e,vk,ns", [
    ([(i, 256, 0) for i in range(9)], 16, 4, 32, 32, False, 1),            # 144 groups of 4 heads: 576 workgroups, by length
    ([(i, 254, 0) for i in range(9)], 16, 4, 32, 36, False, 1),            # the last run of each is short
    ([(i, 250, 0) for i in range(10)], 16, 4, 32, 36, False, 1),           # 63 runs a sequence: groups of two sequences go run by run
    ([(i, 64, 40) for i in range(40)], 16, 4, 20, 20, False, 1),           # all behind 40 keys
    ([(i, 67, 40) for i in range(33)], 16, 4, 32, 32, False, 1),
    ([(i, 120, 0) for i in range(21)] + [(21, 8, 0), (22, 120, 0)], 16, 4, 32, 32, False, 1),
    ([(i, 320, 0) for i in range(3)] + [(3, 319, 1)] + [(i, 320, 0) for i in range(4, 8)], 16, 4, 32, 32, False, 1),      # one begins a position later
    ([(i, 256, 0) for i in range(4)], 8, 8, 64, 64, False, 6),             # 16 groups of 64 rows x 8 heads x 6 splits
    ([(i, 96, 0) for i in range(7)], 16, 1, 72, 64, True, 2),              # values inside keys: groups of 8 rows
    ([(i, 72, 30) for i in range(24)], 16, 1, 40, 40, True, 1),
    ([(i, 33, 70) for i in range(24)], 16, 1, 40, 40, True, 1),
])
def test_equal_sequences(spans, H, G, d, e, vk, ns):
    run(spans, H, G, d, e, 0, 0.0, 0, vk, ns, 700)
