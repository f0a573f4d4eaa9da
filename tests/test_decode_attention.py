"""Decode attention over the paged pool: edges of tiles, pages, partitions and
head groups against float64."""
import pytest
import torch

from llm_d_inference_scheduler_amd.ops import dispatch

KVH, D = 2, 128


@pytest.mark.parametrize("groups", [1, 7, 64, 199, 200, 5000])
@pytest.mark.parametrize("max_len", [1, 31, 256, 257, 5000, 131072])
def test_parts_cover_the_context(groups, max_len):
    parts, part = dispatch.decode_parts(groups, max_len)
    assert 1 <= parts <= 64                   # the kernel's limit
    assert part % 32 == 0                     # parts begin on a page
    assert (parts - 1) * part < max_len <= parts * part


@pytest.mark.parametrize("max_len", [1, 441, 1000, 131072])
@pytest.mark.parametrize("mean", [None, 0.0, 400.0])
@pytest.mark.parametrize("elem", [1, 2])
def test_no_rows(max_len, mean, elem):
    parts, part = dispatch.decode_parts(0, max_len, mean, elem)
    assert 1 <= parts <= 64 and part % 32 == 0
    assert dispatch.decode_waves(0, parts, max_len, mean, elem) in (4, 8)


@pytest.mark.parametrize("groups,max_len,elem,one,several", [
    (136, 8190, 1, 63, 51), (136, 8190, 2, 108, 87), (160, 1875, 2, 27, 34),
    (176, 3750, 2, 54, 58), (96, 1000, 2, 13, 16), (64, 2500, 2, 25, 18),
    (80, 375, 1, 5.9, 8.4), (32, 1250, 2, 13.9, 9.8), (8, 3750, 2, 31, 10),
    (120, 650, 2, 10.3, 15.3), (8, 307, 1, 5.5, 7.8), (24, 6250, 1, 38, 13)])
def test_one_part_or_several(groups, max_len, elem, one, several):
    """Against the times that both took, us."""
    parts, _ = dispatch.decode_parts(groups, max_len, None, elem)
    assert (parts > 1) == (several < one)


@pytest.mark.parametrize("groups,max_len,mean,elem,one,several", [
    (48, 742, 729, 1, 8.7, 9.4), (128, 1874, 1744, 1, 17.3, 20.7),
    (160, 4076, 4076, 1, 34.7, 43.0), (160, 5504, 5168, 1, 43.2, 49.9),
    (8, 777, 777, 2, 11.9, 9.7), (8, 450, 450, 2, 8.7, 9.2),
    (2, 697, 697, 1, 7.9, 8.4), (4, 3300, 3300, 2, 38.9, 10.5),
    (48, 637, 294, 1, 7.5, 9.1), (176, 1205, 488, 1, 12.6, 16.8),
    (80, 1316, 466, 2, 19.3, 12.2), (112, 4323, 3390, 2, 59.1, 43.5),
    (136, 5262, 3223, 2, 70.6, 55.7), (264, 5000, 4000, 2, 125.3, 105.9),
    (320, 625, 500, 2, 22.9, 24.9), (320, 10800, 8000, 2, 270, 241),
    (384, 1875, 1500, 2, 58.0, 58.3), (288, 1250, 1000, 1, 20.6, 24.2),
    (288, 2700, 2000, 1, 40.2, 37.1), (320, 4400, 4000, 1, 66.4, 67.6)])
def test_parts_by_the_mean(groups, max_len, mean, elem, one, several):
    """All lengths alike, or most far below the longest: the bytes follow from the
    mean. Against the times that both took, us."""
    parts, _ = dispatch.decode_parts(groups, max_len, mean, elem)
    assert (parts > 1) == (several < one)


@pytest.mark.parametrize("groups,max_len,elem,one,several", [
    (152, 4993, 2, 72.2, 55.2), (168, 4995, 2, 75.8, 67.2), (136, 3075, 2, 41.9, 37.6),
    (128, 1842, 2, 25.9, 23.3), (128, 3070, 1, 23.9, 20.9), (168, 8741, 1, 66.3, 57.6),
    (160, 8728, 1, 67.7, 62.4), (152, 4993, 1, 37.0, 34.0), (192, 4996, 1, 40.1, 43.2),
    (168, 1873, 2, 28.2, 29.1), (160, 1870, 2, 28.5, 30.1), (136, 1845, 1, 16.3, 18.3)])
def test_one_part_or_several_rounds(groups, max_len, elem, one, several):
    """Lengths a quarter either way. Against the times that both took, us."""
    parts, _ = dispatch.decode_parts(groups, max_len, None, elem)
    assert (parts > 1) == (several < one)


@pytest.mark.parametrize("groups,max_len,mean,elem,eight,four", [
    (256, 374, None, 2, 11.9, 12.1), (256, 374, None, 1, 10.1, 10.2),
    (272, 748, None, 2, 26.7, 25.9), (320, 748, 600, 1, 18.8, 16.6),
    (320, 1871, 1500, 2, 57.0, 52.8), (320, 1871, None, 1, 33.0, 31.0),
    (800, 374, None, 2, 32.4, 28.2), (2048, 624, None, 1, 70.6, 53.3),
    (2048, 1871, None, 2, 252, 257), (800, 150, None, 2, 19, 15),
    (136, 8190, None, 1, 56.5, 51.2), (160, 8700, 7000, 2, 112.9, 105.0),
    (80, 5000, 4000, 2, 32.1, 36.0), (8, 5000, None, 1, 15.0, 15.3),
    (72, 5000, None, 2, 32.4, 32.8), (112, 8700, 7000, 1, 41.6, 43.6),
    (104, 5000, 4000, 2, 45.5, 42.6), (88, 8700, None, 1, 40.3, 36.9)])
def test_waves_of_a_workgroup(groups, max_len, mean, elem, eight, four):
    """Against the times of both, us, in as many parts as each is to have."""
    parts, _ = dispatch.decode_parts(groups, max_len, mean, elem)
    assert dispatch.decode_waves(groups, parts, max_len, mean, elem) == (
        4 if four < eight else 8)


@pytest.mark.parametrize("groups,max_len,mean,elem,eight,four", [
    (288, 2107, 1062, 1, 25.0, 29.6), (608, 8190, 2809, 1, 106, 151),
    (352, 1909, 646, 1, 23.5, 26.4), (424, 1614, 288, 1, 18.7, 22.0),
    (1192, 2412, 1637, 1, 98, 104), (848, 3128, 768, 1, 49.2, 44.8),
    (2072, 2641, 1312, 1, 146, 140), (280, 1348, 296, 2, 20.6, 22.2),
    (408, 672, 378, 2, 21.5, 20.4), (96, 4378, 2855, 2, 36.8, 33.2)])
def test_waves_by_the_mean(groups, max_len, mean, elem, eight, four):
    """Lengths from half as much again as the mean to far apart, as above."""
    parts, _ = dispatch.decode_parts(groups, max_len, mean, elem)
    assert dispatch.decode_waves(groups, parts, max_len, mean, elem) == (
        4 if four < eight else 8)


@pytest.mark.parametrize("batch", [2, 5, 17, 24, 25, 32, 64, 127, 256])
@pytest.mark.parametrize("short", [1, 100, 300, 1000])
@pytest.mark.parametrize("long", [1500, 3000, 8000, 131072])
def test_a_long_sequence_among_short_ones(batch, short, long):
    """No workgroup walks 2000 tokens more than a compute unit's share, and
    batches of like lengths are cut as without their mean."""
    lens = [short] * (batch - 1) + [long]
    mean, groups = sum(lens) / batch, batch * 8
    parts, part = dispatch.decode_parts(groups, long, mean)
    assert 1 <= parts <= 64 and part % 32 == 0
    assert (parts - 1) * part < long <= parts * part
    even = dispatch.decode_parts(groups, long)
    assert parts >= even[0]
    share = sum(lens) * 8 / 256
    assert part <= 1.5 * share + 2000 or parts == 64 or parts < 2 * even[0]
    for like in (short, min(long, 8000)):
        assert dispatch.decode_parts(groups, int(like * 1.25), like) == \
            dispatch.decode_parts(groups, int(like * 1.25))


def _case(lens, qpg, bs, fp8):
    g = torch.Generator().manual_seed(sum(lens) + qpg + bs)
    pages = [-(-n // bs) for n in lens]
    width = max(pages) + 1
    nb = sum(pages) + 1
    dtype = torch.float8_e4m3fn if fp8 else torch.bfloat16
    kc, vc = (torch.randn(nb, KVH, bs, D, generator=g).to(dtype)
              for _ in range(2))
    q = torch.randn(len(lens), KVH * qpg, D, generator=g).bfloat16()
    perm, at = torch.randperm(nb, generator=g).int(), 0
    bt = torch.zeros(len(lens), width, dtype=torch.int32)
    want = torch.zeros(q.shape, dtype=torch.float64)
    for i, (n, p) in enumerate(zip(lens, pages)):
        rows = perm[at:at + p]
        bt[i, :p], at = rows, at + p
        if n == 0:
            continue
        k, v = (c[rows.long()].double().permute(1, 0, 2, 3)
                .reshape(KVH, -1, D)[:, :n] for c in (kc, vc))
        s = q[i].double().view(KVH, qpg, D) @ k.transpose(1, 2) * D ** -0.5
        want[i] = (s.softmax(-1) @ v).view(-1, D)
        if n % bs:                            # the rest of a page is unused
            kc[rows[-1].long(), :, n % bs:] = float("nan")
            vc[rows[-1].long(), :, n % bs:] = float("nan")
    lens = torch.tensor(lens, dtype=torch.int32)
    return [t.cuda() for t in (q, kc, vc, bt, lens)], want


def _close(got, want):
    # half a step of bf16, and the 32-bit sums' error over the context
    torch.testing.assert_close(got.double().cpu(), want, rtol=2 ** -8,
                               atol=1e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("qpg,bs", [(1, 16), (2, 16), (4, 16), (8, 16),
                                    (4, 8), (2, 32), (8, 5)])
@pytest.mark.parametrize("waves", [4, 8])
def test_edges(qpg, bs, fp8, waves):
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    args, want = _case([1, 15, 16, 17, 31, 32, 33, 0, 127, 128, 129, 255, 256,
                        257, 700], qpg, bs, fp8)
    _close(ext.paged_attention(*args, D ** -0.5, waves=waves), want)
    for parts, part in [(3, 256), (64, 11), (8, 96)]:
        _close(ext.paged_attention_split(*args, parts, part, D ** -0.5,
                                         waves=waves), want)


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("batch", [1, 2, 3, 8, 24, 25, 104])
def test_lengths_far_apart(batch, fp8):
    """Every sequence has its parts, whichever order the grid takes them in."""
    lens = [1 + 37 * i % 90 for i in range(batch - 1)] + [2900]
    args, want = _case(lens, 4, 16, fp8)
    mean = sum(lens) / batch
    _close(dispatch.paged_attention(*args, D ** -0.5, 2900, mean), want)
    assert batch == 1 or dispatch.decode_parts(batch * KVH, 2900, mean)[0] > 1
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    for parts, part in [(2, 1472), (12, 256), (64, 48)]:
        for spread in (False, True):
            _close(ext.paged_attention_split(*args, parts, part, D ** -0.5,
                                             spread=spread), want)


@pytest.mark.gpu
def test_attention_of_no_rows():
    (q, *cache, tables, lens), _ = _case([40], 4, 16, False)
    for longest in (None, 40, 1000):
        out = dispatch.paged_attention(q[:0], *cache, tables[:0], lens[:0], D ** -0.5,
                                       longest)
        assert out.shape == (0, KVH * 4, D)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,long,fp8", [(129, 1025, False), (160, 1100, False),
                                            (144, 2049, True)])
def test_a_little_more_than_a_round(batch, long, fp8):
    """In three parts, with the mean length and without, and shorter than said."""
    lens = [long - 61 * i % (long // 4) for i in range(batch)]
    args, want = _case(lens, 4, 16, fp8)
    mean = sum(lens) / batch
    elem = args[1].element_size()
    for m in (mean, None):
        assert dispatch.decode_parts(batch * KVH, long, m, elem)[0] == 3
        assert dispatch.decode_waves(batch * KVH, 3, long, m, elem) == 4
        for said in (long, 3 * long):
            _close(dispatch.paged_attention(*args, D ** -0.5, said, m), want)


@pytest.mark.parametrize("longest,mean,block,page", [
    (1500, None, 16, 25), (1500, 1100.0, 16, 22), (8190, 300.0, 16, 6), (40, None, 16, 0),
    (1500, 1500.0, 5, 100), (1000, 0.0, 16, 0)])
def test_probe(longest, mean, block, page):
    assert dispatch.decode_probe(longest, mean, block) == page


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("bs", [16, 5])
@pytest.mark.parametrize("batch,prefixes", [(2, 1), (7, 3), (65, 64), (66, 65), (150, 4)])
def test_shared_prefixes(batch, prefixes, bs, fp8):
    """However values are read, by the page that is looked at, the sums are the same to
    the bit: rows next to each other that share it, up to 64 and more apart, or none;
    rows that end before it, and one without tokens."""
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    lens = [240 + 37 * i % 90 for i in range(batch)]
    lens[batch // 2] = 0
    lens[-1] = 33
    (q, kc, vc, bt, sl), _ = _case(lens, 4, bs, fp8)
    kc, vc = (c.float().nan_to_num().to(c.dtype) for c in (kc, vc))
    for i in range(prefixes, batch):            # the first 180 tokens
        n = 180 // bs
        bt[i, :n] = bt[i % prefixes, :n]
    args, want = (q, kc, vc, bt, sl, D ** -0.5), []
    for i, n in enumerate(lens):
        k, v = (c[bt[i].long()].double().permute(1, 0, 2, 3).reshape(KVH, -1, D)[:, :n]
                for c in (kc, vc))
        s = q[i].double().view(KVH, 4, D) @ k.transpose(1, 2).contiguous() * D ** -0.5
        want.append((s.softmax(-1) @ v).view(-1, D).cpu())
    want = torch.stack(want)
    for waves in (4, 8):
        whole = ext.paged_attention(*args, waves=waves, probe=-1)
        parted = ext.paged_attention_split(*args[:5], 3, 96, args[5], waves=waves,
                                           spread=True, probe=-1)
        _close(whole, want)
        _close(parted, want)
        for probe in (0, 80 // bs, 180 // bs, 230 // bs, 1 << 20):
            assert torch.equal(whole, ext.paged_attention(*args, waves=waves,
                                                          probe=probe))
            assert torch.equal(parted, ext.paged_attention_split(
                *args[:5], 3, 96, args[5], waves=waves, spread=True, probe=probe))


@pytest.mark.gpu
@pytest.mark.parametrize("qpg,bs", [(1, 16), (8, 16), (4, 5)])
@pytest.mark.parametrize("waves", [4, 8])
def test_values_without_end(qpg, bs, waves):
    """A probability times infinity is infinity, whichever parts the product is
    taken in; two of either sign, or a value that is no number, leave none, and
    other channels keep their sums."""
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    lens = [3, 31, 33, 256, 300, 700]
    args, want = _case(lens, qpg, bs, False)
    vc, bt = args[2], args[3].cpu()
    inf = float("inf")
    for i, n in enumerate(lens):
        for t, channels in [(n // 2, {5: inf, 64: -inf, 100: inf}),
                            (n - 1, {7: -inf, 100: -inf, 127: float("nan")})]:
            for c, x in channels.items():
                vc[int(bt[i, t // bs]), :, t % bs, c] = x
    for c, x in {5: inf, 64: -inf, 7: -inf, 100: float("nan"),
                 127: float("nan")}.items():
        want[:, :, c] = x

    def same(got):
        torch.testing.assert_close(got.double().cpu(), want, rtol=2 ** -8,
                                   atol=1e-4, equal_nan=True)
    same(ext.paged_attention(*args, D ** -0.5, waves=waves))
    for parts, part in [(3, 256), (8, 96)]:
        same(ext.paged_attention_split(*args, parts, part, D ** -0.5,
                                       waves=waves))


@pytest.mark.gpu
def test_running_maximum_far_apart():
    """Scores that grow along the context move the maximum at every tile."""
    args, _ = _case([600], 4, 16, False)
    q, kc, vc, bt, lens = args
    order = bt[0, :38].long()
    for i, page in enumerate(order.tolist()):
        kc[page] = q[0, 0] * (i - 20) * 0.2
    k, v = (c[order].double().permute(1, 0, 2, 3).reshape(KVH, -1, D)[:, :600]
            for c in (kc, vc))
    s = q[0].double().view(KVH, 4, D) @ k.transpose(1, 2).contiguous() \
        * D ** -0.5
    want = (s.softmax(-1) @ v).view(1, -1, D).cpu()
    _close(dispatch.paged_attention(*args, D ** -0.5, 600), want)
    _close(dispatch.paged_attention(*args, D ** -0.5), want)


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("waves", [4, 8])
def test_scores_that_are_no_numbers(fp8, waves):
    """A key that is no number leaves none for the heads that see it, in one part and
    in several; other sequences and heads keep theirs, and one without tokens has 0."""
    from llm_d_inference_scheduler_amd import _hip_ops as ext
    lens, qpg, bs = [700, 3, 0, 257, 33], 4, 16
    args, want = _case(lens, qpg, bs, fp8)
    kc, bt = args[1], args[3].cpu()
    for i, t in ((0, 650), (1, 1), (3, 256)):
        kc[int(bt[i, t // bs]), 1, t % bs, 9] = float("nan")
        want[i, qpg:2 * qpg] = float("nan")

    def same(got):
        torch.testing.assert_close(got.double().cpu(), want, rtol=2 ** -8,
                                   atol=1e-4, equal_nan=True)
    same(ext.paged_attention(*args, D ** -0.5, waves=waves))
    for parts, part in [(3, 256), (8, 96)]:
        same(ext.paged_attention_split(*args, parts, part, D ** -0.5, waves=waves))
