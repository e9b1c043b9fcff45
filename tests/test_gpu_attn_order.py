"""Attention of runs of rows where its workgroups outnumber the places on the chip (their order is then by length), and the join of 2 .. 9 key splits: head sizes that are no
multiple of 4, groups whose last runs are short, sequences that begin inside a group, values inside keys.  The reference is run()'s float64 softmax and its bound: fp32 products
of up to 600 terms and exponentials at 1e-6, 1e-5 of the largest value."""
import pytest

from tests.test_gpu_attn_rows import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spans,H,G,d,e,window,ns", [
    ([(0, 2100, 0)], 16, 4, 32, 32, 0, 1),                                 # 132 groups of 4 head chunks: 528 workgroups, one split
    ([(0, 1203, 0)], 16, 8, 64, 64, 0, 2),                                 # 304 in two splits
    ([(0, 301, 0), (1, 210, 33), (2, 190, 0)], 16, 8, 64, 64, 100, 3),     # 176 in three
    ([(0, 515, 0)], 16, 4, 32, 36, 0, 3),                                  # 396 workgroups: not more than two a CU
])
def test_order(spans, H, G, d, e, window, ns):
    run(spans, H, G, d, e, window, 0.0, 0, False, ns, 2200)


@pytest.mark.parametrize("ns", [2, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("H,G,d,e,vk", [(8, 2, 128, 128, False), (5, 1, 34, 50, False), (6, 2, 20, 9, False), (6, 1, 72, 40, True), (3, 1, 130, 63, True)])
def test_join_of_splits(H, G, d, e, vk, ns):
    run([(0, 67, 300), (1, 9, 0), (2, 130, 0)], H, G, d, e, 0, 0.0, 0, vk, ns, 400)


def test_order_of_values_inside_keys():
    run([(0, 700, 0), (1, 90, 40)], 16, 1, 72, 64, 0, 0.0, 0, True, 2, 800)
