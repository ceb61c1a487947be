"""The rule by which a prompt's attention takes key splits (ops.attention_rows_split) against times of both
forms on an MI355X (us, many rows at once / split passes): the pick is never more than a fifth slower."""

import pytest

# L, nq, nkv, hd, cached, window: many, split
MEASURED = [
    (65, 32, 8, 128, 8000, 0, 358, 77), (255, 32, 8, 128, 8000, 0, 360, 257), (450, 32, 8, 128, 8000, 0, 375, 507),
    (128, 32, 8, 128, 300, 0, 26, 55), (65, 32, 8, 128, 0, 0, 12, 35), (2048, 32, 8, 128, 32000, 0, 1993, 7972),
    (65, 16, 8, 128, 1000, 0, 53, 30), (255, 8, 4, 128, 32000, 0, 1221, 338), (1000, 8, 4, 128, 8000, 0, 321, 563),
    (65, 16, 8, 256, 8000, 0, 585, 120), (200, 16, 8, 256, 16000, 0, 959, 705), (320, 16, 8, 256, 2000, 0, 152, 237),
    (128, 16, 8, 256, 32000, 1024, 76, 119), (1000, 16, 8, 256, 32000, 0, 1942, 7469),
]


@pytest.mark.parametrize("L,nq,nkv,hd,cached,window,many,split", MEASURED)
def test_split_attention_rule(L, nq, nkv, hd, cached, window, many, split):
    from mlx_dspark import ops
    per = ops.attention_rows_split(L, nq, nkv, hd, cached, cached + L + 64, window)
    assert per in (0, 64)
    assert (split if per else many) <= 1.2 * min(many, split)


def test_split_attention_rows_per_pass():
    """As many rows as one split pass takes query rows per kv head, none where a single row has too many."""
    from mlx_dspark import ops
    assert ops.attention_rows_split(65, 64, 8, 128, 16000, 17000) == 32
    assert ops.attention_rows_split(65, 8, 1, 256, 16000, 17000) in (0, 16)
    assert ops.attention_rows_split(65, 257, 1, 128, 16000, 17000) == 0
    assert ops.attention_rows_split(65, 8, 2, 512, 16000, 17000) == 0
