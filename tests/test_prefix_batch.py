"""The batched prefix hash and match against the host's index: lengths around
a wave's 64 blocks, more blocks than are kept, and prompts that are not lists
of plain ints."""
import numpy as np
import pytest
import torch

from llm_d_inference_scheduler_amd import _router_core as rc

pytestmark = pytest.mark.gpu
SEED0 = rc.model_seed("m", "")


@pytest.fixture(scope="module")
def index():
    from llm_d_inference_scheduler_amd.ops.prefix import GpuPrefixIndex
    return GpuPrefixIndex("cuda:0", capacity_pow2=1 << 14)


@pytest.mark.parametrize("block", [1, 7, 16])
@pytest.mark.parametrize("max_blocks", [1, 63, 64, 65, 256, 600])
def test_hashes(index, block, max_blocks):
    rng = np.random.default_rng(block * 1000 + max_blocks)
    blocks = [0, 1, 63, 64, 65, 128, max_blocks, max_blocks + 1]
    prompts = [rng.integers(-2**31, 2**31, n * block + extra).tolist()
               for n in blocks for extra in (0, block - 1)]
    hashes, counts = index.hash_prompts_batch(prompts, block, max_blocks,
                                              SEED0)
    assert hashes.shape == (len(prompts), max_blocks)
    for p, row, n in zip(prompts, hashes.cpu().numpy(), counts.tolist()):
        want = rc.hash_tokens(np.array(p, dtype=np.int32), block, max_blocks,
                              SEED0)
        assert n == len(want)
        assert row[:n].tolist() == want.tolist() and not row[n:].any()


@pytest.mark.parametrize("endpoints", [1, 3, 64, 70])
def test_matches(index, endpoints):
    rng = np.random.default_rng(endpoints)
    host = rc.PrefixIndex(100000)
    tokens = rng.integers(0, 2**31, 16 * 200).astype(np.int32)
    chain = rc.hash_tokens(tokens, 16, 256, SEED0 + endpoints)
    lengths = [0, 1, 63, 64, 65, 128, 129, 200]
    for e in range(0, min(endpoints, 64), 2):      # every other one has some
        part = chain[:lengths[e // 2 % len(lengths)]]
        host.add(e, part)
        index.add(e, part)
    hashes, counts = index.hash_prompts_batch(
        [tokens[:16 * n].tolist() for n in lengths], 16, 256,
        SEED0 + endpoints)
    match = index.match_batch(hashes, counts, endpoints).cpu()
    assert match.shape == (len(lengths), endpoints)
    for row, n in zip(match.tolist(), lengths):
        want = list(host.match_longest(chain[:n], min(endpoints, 64)))
        assert row == want + [0] * (endpoints - 64)


def test_other_prompts(index):
    """What is no list of plain ints goes by way of NumPy, and an int that
    does not fit raises as it does there."""
    ids = list(range(100))
    want = [t.cpu().numpy().tolist()
            for t in index.hash_prompts_batch([ids], 16, 8, SEED0)]
    for prompts in ([tuple(ids)], (ids,), [np.array(ids)],
                    [np.array(ids, dtype=np.int32)],
                    [[np.int64(i) for i in ids]], [[float(i) for i in ids]],
                    [torch.tensor(ids)]):
        got = index.hash_prompts_batch(prompts, 16, 8, SEED0)
        assert [t.cpu().numpy().tolist() for t in got] == want
    for bad in ([2**31], [-2**31 - 1], [2**70]):
        with pytest.raises(OverflowError):
            index.hash_prompts_batch([ids, bad], 16, 8, SEED0)
    hashes, counts = index.hash_prompts_batch([], 16, 8, SEED0)
    assert hashes.shape == (0, 8) and counts.shape == (0,)


def test_ints_of_any_size(index):
    """None, one or two digits of 30 bits, either sign, as NumPy reads them."""
    ids = [0, 1, -1, 255, 256, -256, 2**30 - 1, 2**30, 1 - 2**30, -2**30,
           2**31 - 1, -2**31, 7, 2**15, 2**16, -5] * 3
    want = index.hash_prompts_batch([np.array(ids, dtype=np.int32)], 16, 8,
                                    SEED0)
    got = index.hash_prompts_batch([ids], 16, 8, SEED0)
    assert int(got[1][0]) == 3
    for a, b in zip(got, want):
        assert a.cpu().numpy().tolist() == b.cpu().numpy().tolist()
