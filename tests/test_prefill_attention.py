"""Prefill attention over the paged pool: edges of tiles, pages, heads and
masks, both shapes of the workgroup, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


def _case(seqs, qpg, kvh, bs, fp8, scale):
    """seqs: (new tokens, tokens before). Unused rows of pages hold NaN."""
    g = torch.Generator("cuda").manual_seed(len(seqs) * qpg + bs)

    def draw(*shape):
        return torch.randn(*shape, device="cuda", generator=g)
    pages = [-(-(c + p) // bs) for c, p in seqs]
    dtype = torch.float8_e4m3fn if fp8 else torch.bfloat16
    kc, vc = (draw(sum(pages) + 1, kvh, bs, D).to(dtype) for _ in range(2))
    perm = torch.randperm(sum(pages) + 1, generator=g, device="cuda").int()
    bt = torch.zeros(len(seqs), max(pages), dtype=torch.int32, device="cuda")
    rows = sum(c for c, _ in seqs)
    q = draw(rows, kvh * qpg, D).bfloat16()
    want, size = torch.empty(2, *q.shape, dtype=torch.float64, device="cuda")
    meta, at, row = [], 0, 0
    for i, (c, prior) in enumerate(seqs):
        mine = perm[at:at + pages[i]]
        bt[i, :pages[i]], at = mine, at + pages[i]
        ctx = c + prior
        k, v = (x[mine.long()].double().permute(1, 0, 2, 3)
                .reshape(kvh, -1, D)[:, :ctx] for x in (kc, vc))
        see = torch.arange(ctx, device="cuda") <= prior + torch.arange(
            c, device="cuda")[:, None]
        for h in range(kvh * qpg):
            s = q[row:row + c, h].double() @ k[h // qpg].t().contiguous()
            s = (s * scale).masked_fill(~see, -torch.inf)
            p = s.softmax(-1)
            want[row:row + c, h] = p @ v[h // qpg]
            size[row:row + c, h] = p @ v[h // qpg].abs()
        if ctx % bs:
            for x in (kc, vc):
                x[mine[-1].long(), :, ctx % bs:] = float("nan")
        meta.append((row, c, prior))
        row += c
    tiles = [(i, v) for i, (c, _) in enumerate(seqs)
             for v in range(0, c * qpg, 128)]
    ints = [torch.tensor(t, dtype=torch.int32, device="cuda")
            for t in (meta, tiles)]
    return (q, kc, vc, bt, *ints, scale), (want, size)


def _close(got, want):
    """Probabilities rounded to bf16, at most 2^-8 of each off, so the sum is
    by that share of the same sum of sizes; the result is rounded again."""
    want, size = want
    over = (got.double() - want).abs() - 2 ** -8 * 1.01 * (want.abs() + size)
    assert over.max() < 1e-5


def _as_decoded(got, want):
    """Probabilities of 17 bits, 2^-17 of the sum of sizes, and what 32-bit
    scores and sums add; the result is rounded."""
    want, size = want
    over = (got.double() - want).abs() - 2 ** -8 * 1.01 * want.abs()
    assert (over - 2 ** -15 * size).max() < 1e-5


SEQS = [[(1, 0)], [(1, 700), (31, 0), (32, 1), (33, 31)],
        [(127, 65), (129, 0), (5, 1023)], [(260, 0), (64, 64), (95, 33)]]


@pytest.mark.parametrize("seqs", SEQS)
@pytest.mark.parametrize("qpg,kvh", [(1, 3), (2, 8), (4, 2), (8, 1)])
@pytest.mark.parametrize("bs", [16, 5])
@pytest.mark.parametrize("keys", [0, 1, 2, -1])
def test_pages_in_bf16(seqs, qpg, kvh, bs, keys):
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    args, want = _case(seqs, qpg, kvh, bs, False, D ** -0.5)
    assert args[5].shape[0] * kvh <= 64             # -1: by keys
    (_as_decoded if keys else _close)(ext.flash_prefill(*args, keys=keys),
                                      want)


@pytest.mark.parametrize("bs", [1, 2, 4, 64])
@pytest.mark.parametrize("keys", [0, 1, 2])
def test_sizes_of_pages(bs, keys):
    """Pages of less than a load's four rows, of as many, of a whole tile; last
    tiles of one key, of up to three loads less, and of all."""
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    args, want = _case([(65, 0), (40, 21), (3, 125), (30, 34), (1, 256)], 4, 2,
                       bs, False, D ** -0.5)
    (_as_decoded if keys else _close)(ext.flash_prefill(*args, keys=keys),
                                      want)


@pytest.mark.parametrize("seqs", SEQS)
@pytest.mark.parametrize("qpg,kvh", [(1, 3), (4, 2), (8, 1)])
@pytest.mark.parametrize("bs", [16, 5])
def test_pages_in_fp8(seqs, qpg, kvh, bs):
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    args, want = _case(seqs, qpg, kvh, bs, True, D ** -0.5)
    _close(ext.flash_prefill(*args), want)


@pytest.mark.parametrize("bs", [1, 2, 4, 8, 64, 256])
@pytest.mark.parametrize("fp8", [False, True])
def test_sizes_of_pages_through_registers(bs, fp8):
    """As above; contexts of one to four tiles of keys and one key more or less, waves
    that have seen all of theirs while others have not."""
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    args, want = _case([(65, 0), (40, 21), (3, 125), (30, 34), (1, 256), (128, 0),
                        (191, 1)], 4, 2, bs, fp8, D ** -0.5)
    wide = torch.zeros(7, 1025, dtype=torch.int32, device="cuda")
    wide[:, :args[3].shape[1]] = args[3]
    _close(ext.flash_prefill(*args[:3], wide, *args[4:]), want)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("keys", [0, 1, 2])
@pytest.mark.parametrize("scale", [-0.1, 0.0, 2.0])
def test_scales(fp8, keys, scale):
    """A negative scale turns the order of the scores round, a large one
    moves the maximum at every tile."""
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    args, want = _case([(70, 300), (40, 0)], 4, 2, 16, fp8, scale)
    _close(ext.flash_prefill(*args, keys=keys), want)


def test_long_tables_stage_through_registers():
    """More pages than the table of the direct kernel holds, in bf16."""
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    args, want = _case([(150, 40), (3, 90)], 4, 2, 16, False, D ** -0.5)
    wide = torch.zeros(2, 1025, dtype=torch.int32, device="cuda")
    wide[:, :args[3].shape[1]] = args[3]
    _close(ext.flash_prefill(*args[:3], wide, *args[4:]), want)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("keys", [0, 1, 2])
@pytest.mark.parametrize("pages", [0, 1025])
def test_scores_that_are_no_numbers(fp8, keys, pages):
    """A key that is no number leaves none for the rows and heads that see it, and every
    row is written."""
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    seqs = [(70, 300), (40, 0), (3, 65)]
    args, (want, size) = _case(seqs, 4, 2, 16, fp8, D ** -0.5)
    tables, row = args[3], 0
    for i, ((n, prior), t) in enumerate(zip(seqs, (350, 0, 67))):
        args[1][tables[i, t // 16].long(), 1, t % 16, 9] = float("nan")
        want[row + max(0, t - prior):row + n, 4:] = float("nan")
        row += n
    if pages:
        tables = torch.zeros(3, pages, dtype=torch.int32, device="cuda")
        tables[:, :args[3].shape[1]] = args[3]
    for _ in range(3):
        torch.full_like(args[0], 3.0)          # what an unwritten row would hold
        got = ext.flash_prefill(*args[:3], tables, *args[4:], keys=keys)
        none = want.isnan()
        assert got[none].isnan().all()
        _close(got[~none], (want[~none], size[~none]))


@pytest.mark.parametrize("bs", [1, 16])
@pytest.mark.parametrize("seqs", [[(1, 0)], [(3, 90), (64, 1)], [(150, 40), (1, 300)]])
def test_an_infinite_value_through_registers(seqs, bs):
    """The last key of each prompt has infinite values: infinity for its last query,
    which sees it, however far the tile goes on behind it."""
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    args, want = _case(seqs, 4, 2, bs, False, D ** -0.5)
    q, kc, vc, tables = args[:4]
    last, at = [], 0
    for i, (n, prior) in enumerate(seqs):
        t = n + prior - 1
        vc[tables[i, t // bs].long(), :, t % bs, 5] = torch.inf
        vc[tables[i, t // bs].long(), :, t % bs, 100] = -torch.inf
        at += n
        last.append(at - 1)
    wide = torch.zeros(len(seqs), 1025, dtype=torch.int32, device="cuda")
    wide[:, :tables.shape[1]] = tables
    got = ext.flash_prefill(q, kc, vc, wide, *args[4:])[last]
    assert (got[..., 5] == torch.inf).all() and (got[..., 100] == -torch.inf).all()
    rest = [c for c in range(D) if c not in (5, 100)]
    _close(got[..., rest], [x[last][..., rest] for x in want])


@pytest.mark.parametrize("seqs,qpg,kvh", [
    ([(300, 0)], 4, 8), ([(400, 300)], 4, 8), ([(100, 40)] * 4, 4, 8),
    ([(20, 300)] * 12, 4, 8), ([(250, 0)], 8, 8), ([(900, 0)], 4, 8),
    ([(500, 0), (100, 600)], 4, 8), ([(1020, 0)], 1, 16)])
def test_workgroups_fewer_than_compute_units(seqs, qpg, kvh):
    """64 to 255 workgroups by rows: both shapes, and the one that is taken,
    are as exact as decoding."""
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    from llm_d_inference_scheduler_amd import ops
    args, want = _case(seqs, qpg, kvh, 16, False, D ** -0.5)
    assert 64 < args[5].shape[0] * kvh < 256
    shape = ops.prefill_shape([n for n, _ in seqs], [n + p for n, p in seqs],
                              qpg, kvh)
    assert shape in (1, 2)
    for keys in (1, 2, shape, -1):
        _as_decoded(ext.flash_prefill(*args, keys=keys), want)
    plain = ext.flash_prefill(*args, keys=0)       # rounded to bf16
    _close(plain, want)
    with pytest.raises(AssertionError):
        _as_decoded(plain, want)
