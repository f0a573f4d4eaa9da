"""Which products of few rows the framework's kernels take, by the sizes: where both
sides were timed, the faster one. On the CPU, through the rules' C entries."""
import ctypes

import pytest
import torch  # noqa: F401  (the extension's libraries)

from llm_d_inference_scheduler_amd import _hip_layered

RULES = ctypes.CDLL(_hip_layered.__file__)
EVERY = (1, 16, 17, 24, 32, 33, 48, 64)


# rows of x by which the library and the activation are slower
@pytest.mark.parametrize("n,k,rows", [
    (64, 2048, EVERY), (256, 2560, EVERY), (192, 2800, EVERY), (520, 3072, EVERY),
    (512, 3584, (1, 16)), (520, 3392, (1, 16)), (64, 4096, (1, 16)),
    (768, 4096, EVERY[:5]), (1296, 3840, EVERY), (1024, 4096, EVERY),
    (2048, 4608, EVERY), (2336, 4712, EVERY), (2336, 6096, EVERY),
    (64, 5120, ()), (1536, 5120, ()), (2048, 5120, EVERY[:5]), (3072, 5632, EVERY[:6]),
    (4096, 5120, EVERY), (2048, 6144, EVERY[:5]), (2048, 7168, ()),
    (3072, 7168, EVERY[:5]), (4096, 7680, EVERY), (4096, 8192, (1, 16)),
    (8000, 8192, (1, 16)), (14336, 4096, EVERY), (8704, 10240, EVERY)])
def test_gated(n, k, rows):
    taken = [m for m in EVERY if RULES.lds_linear_rows_takes(m, n, k, 1, 0)]
    assert taken == list(rows)


# rows of x by which parts and their sum are slower than one part
@pytest.mark.parametrize("n,k,rows", [
    (8, 2048, EVERY), (1024, 4096, (1, 16)), (2048, 3072, EVERY[:5]),
    (2304, 4096, (1, 16)), (2560, 3840, (1, 16)), (3072, 3072, EVERY),
    (3072, 4096, EVERY[:5]), (3000, 3992, EVERY[:5]), (2048, 8192, (1, 16)), (4096, 5120, (1, 16)),
    (8192, 4096, EVERY), (10240, 3584, EVERY), (10240, 4096, EVERY[:5]),
    (8192, 5120, EVERY[:5]), (8192, 7680, EVERY[:5]), (8192, 8192, EVERY),
    (8192, 8184, EVERY[:5]),
    (9216, 4608, EVERY), (9216, 7680, EVERY), (9216, 8192, EVERY[:5]), (10240, 6144, EVERY[:5]), (12800, 8192, EVERY),
    (16384, 5120, EVERY)])
def test_one_part(n, k, rows):
    assert [m for m in EVERY if RULES.lds_linear_plain_parts(m, n, k) == 1] == list(rows)


def test_an_index_of_another_device_is_no_index():
    """The kernels read one by its address; torch's own says what is wrong with it."""
    from llm_d_inference_scheduler_amd.ops.dispatch import _index
    table, ids = torch.zeros(4, 8), torch.zeros(6, dtype=torch.int64)
    assert _index(ids, table)
    for other in (ids.to("meta"), ids.int(), ids[::2], ids.view(2, 3)):
        assert not _index(other, table)
