"""Which shape of workgroups takes a prefill attention call, against the times
that both took (us: by keys, by rows with 17 bits)."""
import pytest

from llm_d_inference_scheduler_amd import ops

# prompts (new tokens, tokens before), heads per key head, key heads, times
TIMED = [
    ([(1200, 0)], 4, 2, 26, 54), ([(1200, 1000)], 1, 8, 52, 86),
    ([(1200, 4000)], 1, 8, 137, 195), ([(300, 0)], 4, 8, 13.0, 17.7),
    ([(300, 1000)], 4, 8, 44, 55), ([(300, 4000)], 4, 8, 130, 164),
    ([(150, 300)], 8, 8, 20.7, 23.4), ([(20, 0)] * 12, 4, 8, 12.7, 6.7),
    ([(20, 2000)] * 12, 4, 8, 72, 81), ([(60, 0)] * 6, 4, 8, 13.0, 8.5),
    ([(400, 300)], 4, 8, 26.5, 34.3), ([(200, 2000)] * 2, 4, 8, 78, 89),
    ([(150, 0)] * 3, 4, 8, 14.6, 12.5), ([(100, 0)] * 4, 4, 8, 12.8, 9.9),
    ([(500, 1000)], 4, 8, 52, 66), ([(600, 4000)], 4, 8, 195, 175),
    ([(300, 1000)], 8, 8, 69, 59), ([(300, 500)] * 2, 4, 8, 45, 39),
    ([(500, 0), (100, 3000)], 4, 8, 56, 122), ([(700, 4000)], 4, 8, 200, 183),
    ([(50, 500)] * 12, 4, 8, 43, 29), ([(800, 1000)], 4, 8, 101, 79),
    ([(200, 500)] * 4, 4, 8, 56, 36), ([(450, 0)] * 2, 4, 8, 36, 27)]


@pytest.mark.parametrize("seqs,group,heads,keys,rows", TIMED)
def test_the_faster_one(seqs, group, heads, keys, rows):
    news, ctxs = [n for n, _ in seqs], [n + p for n, p in seqs]
    assert ops.prefill_shape(news, ctxs, group, heads) == \
        (1 if keys < rows else 2)


def test_few_and_many_workgroups():
    assert ops.prefill_shape([], [], 4, 8) == 1
    assert ops.prefill_shape([1], [1], 8, 1) == 1
    assert ops.prefill_shape([256], [5000], 4, 8) == 1     # 256 by keys
    assert ops.prefill_shape([993], [1993], 4, 8) == 0     # 256 by rows
    assert ops.prefill_shape([8000], [8000], 4, 8) == 0
