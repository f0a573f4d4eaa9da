"""Ops of grouped attention, experts and the looped stream one by one against
the plain oracle: the CPU versions everywhere, the HIP kernels in both
precisions on a GPU."""
import pytest
import torch

import sezazen_oracle as oracle
from llm_d_inference_scheduler_amd.ops import layered as ops
from llm_d_inference_scheduler_amd.ops.dispatch import decode_parts, decode_waves
from test_layered_ops import F64, GPU, RUNS, close, f64, meta, put, rnd

F32 = ("", torch.float32)


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("width", [38, 64, 1000, 4096, 9000])
class TestStream:
    def test_embedding_with_positions(self, run, width):
        table, pos = put(rnd(11, width), run), rnd(9, width, seed=4)
        ids = torch.tensor([3, 0, 10, 3], device=run[0])
        at = torch.tensor([0, 8, 3, 7], dtype=torch.int32, device=run[0])
        wn = rnd(width, seed=3)
        want = f64(table)[ids.cpu()] * 2.5 + pos.double()[at.cpu().long()]
        x, h = ops.embed_norm(ids, table, 2.5, wn.to(run[0]), 0.0, 1e-3,
                              pos.to(run[0]), at)
        assert x.dtype == torch.float32
        assert (f64(x) - want).abs().max() < 1e-5
        close(h, oracle.rms_norm(want, wn.double(), 1e-3), run)
        x, h = ops.embed_norm(ids, table, 2.5, None, 0.0, 1e-3,
                              pos.to(run[0]), at)      # no norm: a copy
        assert torch.equal(h, x.to(run[1]))

    @pytest.mark.parametrize("n", [0, 1, 3])
    @pytest.mark.parametrize("has_y", [True, False])
    def test_sum(self, run, width, n, has_y):
        x, y = rnd(5, width), put(rnd(5, width, seed=1), run)
        rows = put(rnd(5 * n, width, seed=2), run) if n else None
        wn = rnd(width, seed=3)
        xd = x.clone().to(run[0])
        h = ops.stream_norm(xd, y if has_y else None, None, wn.to(run[0]),
                            0.0, 1e-3, run[1], rows)
        want = x.double()
        if has_y:
            want = want + f64(y)
        if n:
            want = want + f64(rows).view(5, n, width).sum(1)
        assert (f64(xd) - want).abs().max() < 3e-6      # stays 32-bit
        close(h, oracle.rms_norm(want, wn.double(), 1e-3), run)
        h = ops.stream_norm(xd, None, None, None, 0.0, 1e-3, run[1])
        assert torch.equal(h, xd.to(run[1]))

    def test_loop_entry(self, run, width):
        a, b, v = rnd(5, width), rnd(5, width, seed=1), rnd(width, seed=2)
        wn = rnd(width, seed=3)
        x = torch.full((5, width), float("nan"), device=run[0])
        h = ops.loop_norm(x, a.to(run[0]), b.to(run[0]), v.to(run[0]),
                          wn.to(run[0]), 0.0, 1e-3, run[1])
        want = a.double() + b.double() + v.double()
        assert (f64(x) - want).abs().max() < 3e-6
        close(h, oracle.rms_norm(want, wn.double(), 1e-3), run)


@pytest.mark.parametrize("run", RUNS)
class TestActivations:
    @pytest.mark.parametrize("size", [22, 64])
    def test_silu_gate(self, run, size):
        gu = put(rnd(7, 2 * size, scale=4), run)
        gu[0, 0], gu[0, 1] = 90.0, -90.0
        close(ops.gated_act(gu, "silu"),
              oracle.silu(f64(gu)[:, :size]) * f64(gu)[:, size:], run)

    @pytest.mark.parametrize("size", [22, 64])
    def test_relu_squared(self, run, size):
        x = put(rnd(7, size, scale=4), run)
        close(ops.activate(x, "relu_squared"), oracle.relu_squared(f64(x)),
              run)

    def test_linear32(self, run):
        x, w = put(rnd(33, 72), run), put(rnd(40, 72, seed=1), run)
        y = ops.linear32(x, w)
        assert y.dtype == torch.float32
        close(y, f64(x) @ f64(w).T, F32, f32=2e-6)


# ---- grouped attention ------------------------------------------------------
BS = 16


def paged(run, G, D, V, ctxs, seed=0):
    """-> cache with scattered pages, block tables, [(k, v)] in 64-bit. Pages
    that no sequence owns hold values that would show."""
    blocks = sum(-(-c // BS) for c in ctxs) + 3
    g = torch.Generator().manual_seed(seed)
    order = torch.randperm(blocks, generator=g).tolist()
    cache = torch.full((blocks, G, BS, D + V), 50.0)
    tables = torch.zeros(len(ctxs), max(-(-c // BS) for c in ctxs) + 1,
                         dtype=torch.int32)
    kv = []
    for s, c in enumerate(ctxs):
        k, v = rnd(c, G, D, seed=seed + s), rnd(c, G, V, seed=seed + 50 + s)
        k, v = k.to(run[1]), v.to(run[1])
        kv.append([k.double(), v.double()])
        for t in range(c):
            if t % BS == 0:
                tables[s, t // BS] = order.pop()
            cache[tables[s, t // BS], :, t % BS] = torch.cat(
                [k[t], v[t]], -1).float()
    return put(cache, run), tables.to(run[0]), kv


def expected(q, k, v, pos, scale, sink):
    """q [H, D] at position pos; k [T, G, D], v [T, G, V] -> [H V]."""
    H, G = q.shape[0], k.shape[1]
    out = []
    for h in range(H):
        g = h // (H // G)
        s = (k[:pos + 1, g] @ q[h] * scale)[None]
        see = torch.ones_like(s, dtype=torch.bool)
        p = oracle.sink_softmax(s, see) if sink is not None \
            else torch.softmax(s, -1)
        out.append(p @ v[:pos + 1, g])
    return torch.cat(out, -1)[0]


# H, G, D, V: vector and odd sizes, one to many heads per group
HEADS = [(4, 2, 16, 24), (6, 1, 24, 8), (3, 3, 7, 5), (20, 1, 40, 72),
         (8, 2, 128, 128), (33, 1, 64, 16), (4, 2, 192, 256), (2, 1, 12, 40)]


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("H,G,D,V", HEADS)
class TestGroupedAttention:
    def test_store(self, run, H, G, D, V):
        proj = put(rnd(7, H * D + G * (D + V) + 8), run)
        cache = put(torch.full((4, G, BS, D + V), 9.0), run)
        before = cache.clone()
        slots = torch.tensor([3, 60, 15, 16, 17, 0, 63], device=run[0])
        ops.store_heads(proj, H * D, slots, cache, D)
        for i, s in enumerate(slots.tolist()):
            got = cache[s // BS, :, s % BS]
            split = H * D + G * D
            assert torch.equal(got[:, :D].flatten(),
                               proj[i, H * D:split])
            assert torch.equal(got[:, D:].flatten(),
                               proj[i, split:split + G * V])
            before[s // BS, :, s % BS] = got
        assert torch.equal(cache, before)

    @pytest.mark.parametrize("plain", [False, True])
    @pytest.mark.parametrize("sink", [0.0, None, 1.5])
    def test_decode(self, run, H, G, D, V, plain, sink):
        if sink == 1.5:
            def want_row(q, k, v, pos):     # exp(1.5) in the sum
                k2 = torch.cat([torch.zeros_like(k[:1]), k])
                v2 = torch.cat([torch.zeros_like(v[:1]), v])
                out = []
                for h in range(H):
                    g = h // (H // G)
                    s = k2[:pos + 2, g] @ q[h] * scale
                    s[0] = 1.5
                    out.append(torch.softmax(s, -1) @ v2[:pos + 2, g])
                return torch.cat(out)
        else:
            def want_row(q, k, v, pos):
                return expected(q, k, v, pos, scale, sink)
        ctxs = [1, 2, 15, 16, 17, 63, 64, 65, 129, 300, 700]
        if plain:
            ctxs = [1, 17, 300]
        scale = 1.2 * D ** -0.5
        cache, tables, kv = paged(run, G, D, V, ctxs)
        n = len(ctxs)
        proj = put(rnd(n + 2, H * D + G * (D + V), seed=3), run)
        pos = torch.tensor([c - 1 for c in ctxs] + [0, 0], dtype=torch.int32)
        seq = torch.arange(n + 2, dtype=torch.int32)
        out = put(torch.full((n + 2, H * V), 7.0), run)
        ops.grouped_decode(proj, cache, pos.to(run[0]), seq.to(run[0]),
                           tables, n, H, D, scale, sink, max(ctxs), out,
                           plain=plain)
        q = f64(proj)[:, :H * D].view(n + 2, H, D)
        want = torch.stack([want_row(q[i], *kv[i], ctxs[i] - 1)
                            for i in range(n)])
        close(out[:n], want, run, f32=5e-6)
        assert (out[n:] == 7).all()

    @pytest.mark.parametrize("plain", [False, True])
    @pytest.mark.parametrize("sink", [0.0, None])
    def test_prefill(self, run, H, G, D, V, plain, sink):
        """Portions with and without earlier tokens, around tile sizes."""
        portions = [(0, 64), (17, 70), (200, 9), (63, 130)]
        if plain:
            portions = [(0, 20), (17, 9)]
        scale = 1.2 * D ** -0.5
        cache, tables, kv = paged(run, G, D, V, [a + n for a, n in portions])
        base = 3        # decoded rows in front: not touched
        seqs, pos = [], [0] * base
        for i, (prior, n) in enumerate(portions):
            seqs.append((n, prior, 0))
            pos += range(prior, prior + n)
        m, rows = meta(seqs, run)
        m[:, 0] += base
        rows = torch.cat([torch.zeros_like(rows[:base]), rows])
        T = base + sum(n for _, n in portions)
        per = max(1, 128 * G // H)
        tiles = torch.tensor([(i, r) for i, (_, n) in enumerate(portions)
                              for r in range(0, n, per)], dtype=torch.int32)
        proj = put(rnd(T, H * D + G * (D + V), seed=3), run)
        out = put(torch.full((T, H * V), 7.0), run)
        ops.grouped_prefill(
            proj, cache, torch.tensor(pos, dtype=torch.int32).to(run[0]),
            rows, tables, base, m, tiles.to(run[0]), H, D, scale, sink, out,
            plain=plain)
        q = f64(proj)[:, :H * D].view(T, H, D)
        want, row = [], base
        for (prior, n), (k, v) in zip(portions, kv):
            for t in range(n):
                want.append(expected(q[row], k, v, prior + t, scale, sink))
                row += 1
        close(out[base:], torch.stack(want), run, f32=5e-6)
        assert (out[:base] == 7).all()

    def test_one_key_stands_out(self, run, H, G, D, V):
        """A key far back, at page and tile borders, and the token's own: the
        output is that key's value, in decoding and in a portion. The key
        after the query would win as well if it were seen."""
        ctx = 520
        for at in (0, 15, 16, 63, 64, 128, 447, 448, 511, 518):
            cache, tables, kv = paged(run, G, D, V, [ctx], seed=at)
            k, v = kv[0]
            strong = 40.0 * torch.ones(D, dtype=F64) / D ** 0.5
            for t, x in ((at, strong), (519, 1.5 * strong)):
                blk = tables[0, t // BS]
                cache[blk, :, t % BS, :D] = x.to(cache)
            q = torch.ones(1, H, D) / D ** 0.5
            proj = torch.cat([q.flatten(1), torch.zeros(1, G * (D + V))], 1)
            want = torch.cat([v[at, h // (H // G)] for h in range(H)])
            for n in (1, 200):      # one row; the last of a portion
                T, prior = n, 519 - n
                p = put(proj.expand(T, -1), run)
                pos = torch.arange(prior, prior + n, dtype=torch.int32,
                                   device=run[0])
                seq = torch.zeros(T, dtype=torch.int32, device=run[0])
                out = put(torch.zeros(T, H * V), run)
                if n == 1:
                    ops.grouped_decode(p, cache, pos, seq, tables, 1, H, D,
                                       1.0, 0.0, 519, out)
                else:
                    m, _ = meta([(n, prior, 0)], run)
                    per = max(1, 128 * G // H)
                    tiles = torch.tensor([(0, r) for r in range(0, n, per)],
                                         dtype=torch.int32, device=run[0])
                    ops.grouped_prefill(p, cache, pos, seq, tables, 0, m,
                                        tiles, H, D, 1.0, 0.0, out)
                close(out[-1], want, run, f32=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("parts", [1, 2, 5, 8, 9])
@pytest.mark.parametrize("rows,H,G,D,V,extra", [
    (1, 4, 2, 128, 128, 0), (7, 3, 3, 8, 16, 8), (33, 2, 1, 40, 8, 0),
    (60, 32, 8, 128, 128, 0)])
def test_store_of_parts(parts, rows, H, G, D, V, extra):
    """The sums in 32 bits, part by part, and one rounding: to the bit."""
    run = ("cuda", torch.bfloat16)
    part = rnd(parts, rows, H * D + G * (D + V) + extra, seed=parts).cuda()
    total = part[0].clone()
    for p in part[1:]:
        total += p
    want = put(torch.full((rows // BS + 2, G, BS, D + V), 9.0), run)
    cache = want.clone()
    slots = torch.randperm(rows + 3, generator=torch.Generator().manual_seed(rows))
    slots = slots[:rows].cuda()
    ops.store_heads(total.bfloat16(), H * D, slots, want, D)
    q = ops.store_heads(part, H * D, slots, cache, D)
    assert torch.equal(cache, want)
    assert torch.equal(q, total.bfloat16()[:, :H * D])


@pytest.mark.gpu
@pytest.mark.parametrize("rep", [1, 3, 8])
@pytest.mark.parametrize("bs", [16, 5])
@pytest.mark.parametrize("sink", [0.0, None])
@pytest.mark.parametrize("ctxs", [
    [1, 31, 32, 33, 200, 256], [257, 1, 40], [3, 2000, 1025, 512], [130, 1] * 34])
def test_decode_of_heads_of_128(rep, bs, sink, ctxs, monkeypatch):
    """Four and eight waves, one part and several, of rows that have fewer tokens than
    parts; tiles' and pages' ends."""
    monkeypatch.setitem(globals(), "BS", bs)
    run, G, D = ("cuda", torch.bfloat16), 3, 128
    H, n = rep * G, len(ctxs)
    cache, tables, kv = paged(run, G, D, D, ctxs)
    proj = put(rnd(n, H * D + 2 * G * D, seed=3), run)
    pos = torch.tensor([c - 1 for c in ctxs], dtype=torch.int32, device="cuda")
    seq = torch.arange(n, dtype=torch.int32, device="cuda")
    out = put(torch.full((n, H * D), 7.0), run)
    scale = 1.2 * D ** -0.5
    ops.grouped_decode(proj, cache, pos, seq, tables, n, H, D, scale, sink, max(ctxs),
                       out)
    q = f64(proj)[:, :H * D].view(n, H, D)
    want = torch.stack([expected(q[i], *kv[i], c - 1, scale, sink)
                        for i, c in enumerate(ctxs)])
    # probabilities have 24 bits: 32-bit scores and sums, and the result's rounding
    assert ((f64(out) - want).abs() <= 2 ** -8 * want.abs() + 2e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 4, 70])
def test_rows_of_one_sequence(rows, monkeypatch):
    """They read one table: the same bits by whichever page that is found, if at all."""
    run, G, D, H = ("cuda", torch.bfloat16), 3, 128, 6
    ctxs = [300, 120]
    cache, tables, kv = paged(run, G, D, D, ctxs)
    n = 2 * rows
    proj = put(rnd(n, H * D, seed=4), run)
    pos = torch.tensor([c - rows + i for c in ctxs for i in range(rows)],
                       dtype=torch.int32, device="cuda")
    seq = torch.tensor([i for i in (0, 1) for _ in range(rows)], dtype=torch.int32,
                       device="cuda")
    outs = []
    for probe in (-1, 0, 6, 9, 1 << 20):
        monkeypatch.setattr(ops, "decode_probe", lambda *a: probe)
        outs.append(put(torch.zeros(n, H * D), run))
        ops.grouped_decode(proj, cache, pos, seq, tables, n, H, D, D ** -0.5, None, 300,
                           outs[-1])
    q = f64(proj).view(n, H, D)
    want = torch.stack([expected(q[i], *kv[i // rows], int(pos[i]), D ** -0.5, None)
                        for i in range(n)]).view(n, -1)
    assert all(torch.equal(o, outs[0]) for o in outs)
    assert ((f64(outs[0]) - want).abs() <= 2 ** -8 * want.abs() + 2e-5).all()


@pytest.mark.parametrize("n,longest,mean", [
    (12, 5000, None), (12, 5000, 3400.0), (12, 5000, 2100.0), (12, 5000, 1900.0),
    (33, 900, None), (33, 900, 300.0), (33, 3000, 2500.0), (16, 3000, 2800.0)])
def test_waves_of_decode(monkeypatch, n, longest, mean):
    """The kernel is told what the rule says; shares of every row up to 2.5 times the
    mean."""
    told = []
    monkeypatch.setattr(ops.ref, "grouped_decode",
                        lambda *a: told.append(a[-3:]))
    cache = torch.zeros(1, 8, 16, 256)
    ops.grouped_decode(torch.zeros(n, 32 * 128), cache, None, None, None, n, 32, 128,
                       1.0, None, longest, None, mean_ctx=mean)
    parts, tokens = decode_parts(n * 8, longest, mean)
    far = mean is not None and longest > 2.5 * mean
    assert told == [(parts, tokens if far else 0, decode_waves(
        n * 8, parts, longest, mean, apart=2.5))]


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("mean", [None, 100.0])
def test_decode_of_no_rows(run, D, mean):
    cache, tables, _ = paged(run, 2, D, D, [40])
    for rows in (0, 3):                 # of them none of one token
        out = put(torch.full((rows, 4 * D), 7.0), run)
        seq = torch.zeros(rows, dtype=torch.int32, device=run[0])
        ops.grouped_decode(put(rnd(rows, 4 * D, seed=3), run), cache, seq, seq,
                           tables if rows else tables[:0], 0, 4, D, D ** -0.5, None,
                           1000, out, mean_ctx=mean)
        assert (out == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("G,rep,ctxs", [
    (8, 2, [80 + 11 * i % 90 for i in range(14)] + [1421]),      # 5 parts
    (4, 4, [9 + 7 * i % 300 for i in range(34)] + [1770]),       # 4
    (2, 1, [1 + 37 * i % 90 for i in range(103)] + [2900])])     # 10: by the longest
@pytest.mark.parametrize("sink", [0.0, None])
def test_decode_of_rows_far_apart(G, rep, ctxs, sink):
    """One long row among short ones is in parts where the mean is known."""
    run, D = ("cuda", torch.bfloat16), 128
    H, n, mean = rep * G, len(ctxs), sum(ctxs) / len(ctxs)
    assert decode_parts(n * G, max(ctxs), mean)[0] > decode_parts(n * G, max(ctxs))[0]
    cache, tables, kv = paged(run, G, D, D, ctxs)
    proj = put(rnd(n, H * D, seed=3), run)
    pos = torch.tensor([c - 1 for c in ctxs], dtype=torch.int32, device="cuda")
    seq = torch.arange(n, dtype=torch.int32, device="cuda")
    q = f64(proj).view(n, H, D)
    want = torch.stack([expected(q[i], *kv[i], c - 1, D ** -0.5, sink)
                        for i, c in enumerate(ctxs)])
    for said in (max(ctxs), max(ctxs) - 300):      # the longest, or less
        out = put(torch.full((n, H * D), 7.0), run)
        ops.grouped_decode(proj, cache, pos, seq, tables, n, H, D, D ** -0.5, sink, said,
                           out, mean_ctx=mean)
        # as test_decode_of_heads_of_128
        assert ((f64(out) - want).abs() <= 2 ** -8 * want.abs() + 2e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("sink", [0.0, None])
@pytest.mark.parametrize("ctxs", [[40, 257, 1, 600], [3, 2000], [33] * 90])
def test_scores_that_are_no_numbers(D, sink, ctxs):
    """A key that is no number or infinite leaves no number for the heads that see it;
    keys that are all infinitely far leave none, or a sink all. Other heads and rows
    keep theirs."""
    run, G, rep = ("cuda", torch.bfloat16), 3, 4
    H, n = rep * G, len(ctxs)
    cache, tables, kv = paged(run, G, D, D, ctxs)
    proj = put(rnd(n, H * D + 2 * G * D, seed=3), run)
    proj[:, 0:H * D:D] = 1.0                  # channel 0 of all queries
    table = tables.cpu()

    def key(i, t, g, x):
        cache[int(table[i, t // BS]), g, t % BS, 0] = x
    key(0, ctxs[0] // 2, 0, float("nan"))
    key(1, ctxs[1] - 1, 1, float("inf"))
    for t in range(ctxs[-1]):
        key(n - 1, t, 2, -float("inf"))
    pos = torch.tensor([c - 1 for c in ctxs], dtype=torch.int32, device="cuda")
    seq = torch.arange(n, dtype=torch.int32, device="cuda")
    out = put(torch.full((n, H * D), 7.0), run)
    ops.grouped_decode(proj, cache, pos, seq, tables, n, H, D, D ** -0.5, sink, max(ctxs),
                       out)
    got, q = f64(out).view(n, G, rep, D), f64(proj)[:, :H * D].view(n, H, D)
    assert got[0, 0].isnan().all() and got[1, 1].isnan().all()
    if sink is not None:
        assert (got[-1, 2] == 0).all()
    elif D == 128:
        assert got[-1, 2].isnan().all()
    want = torch.stack([expected(q[i], *kv[i], c - 1, D ** -0.5, sink)
                        for i, c in enumerate(ctxs)]).view(n, G, rep, D)
    for i, g in ((0, 0), (1, 1), (n - 1, 2)):
        got[i, g] = want[i, g] = 0
    close(got, want, run, f32=1e-5)


# ---- experts ----------------------------------------------------------------
@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("T,K,E,top", [
    (1, 38, 5, 2), (17, 64, 3, 3), (40, 200, 16, 1), (33, 64, 33, 8),
    (5, 72, 100, 4), (16, 128, 256, 7), (9, 64, 300, 2)])
class TestRoute:
    def test_choice_and_scores(self, run, T, K, E, top):
        h, w = put(rnd(T, K), run), put(rnd(E, K, seed=1, scale=K ** -0.5),
                                        run)
        ids, wt = ops.route(h, w, top)
        assert ids.dtype == torch.int32 and wt.dtype == torch.float32
        want_ids, want = oracle.route(f64(h), f64(w), top)
        # sums differ in order only: scores agree, and so do clear choices
        close(wt, want, F32, f32=1e-5)
        s = oracle.sigmoid(f64(h) @ f64(w).T)
        ids = ids.cpu().long()
        assert all(len(set(r)) == top for r in ids.tolist())
        assert (torch.gather(s, 1, ids) - want).abs().max() < 1e-5

    def test_ties_go_to_the_lower_expert(self, run, T, K, E, top):
        h, w = put(rnd(T, K), run), put(torch.zeros(E, K), run)
        ids, wt = ops.route(h, w, top)
        assert ids.tolist() == [list(range(top))] * T
        assert (wt == 0.5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 16, 31])
@pytest.mark.parametrize("K,E,top", [
    (1024, 16, 2), (2056, 7, 2), (1160, 17, 4), (1016, 32, 4), (640, 33, 8),
    (520, 64, 8), (504, 65, 8), (1032, 128, 8), (264, 129, 3), (248, 255, 9)])
def test_route_by_groups_of_experts(T, K, E, top):
    """Each split of experts and K over waves: whole steps, remainders of 8, waves
    without a step, rows and experts past the end."""
    run = ("cuda", torch.bfloat16)
    h, w = put(rnd(T, K), run), put(rnd(E, K, seed=1, scale=K ** -0.5), run)
    ids, wt = ops.route(h, w, top)
    want_ids, want = oracle.route(f64(h), f64(w), top)
    # sums of K products of size K ** -0.5 in 32 bits, then a slope of at most 1/4:
    # under K * 2 ** -24 * 8 / K ** 0.5 / 4 < 6e-6
    assert (wt.cpu().double() - want).abs().max() < 6e-6
    s = oracle.sigmoid(f64(h) @ f64(w).T)
    assert (torch.gather(s, 1, ids.cpu().long()) - want).abs().max() < 6e-6


@pytest.mark.gpu
@pytest.mark.parametrize("T", [3, 4, 5, 1023, 1024, 1025])
@pytest.mark.parametrize("K,E,top", [(136, 32, 4), (512, 130, 8)])
def test_route_by_4_and_16_rows(T, K, E, top):
    run = ("cuda", torch.bfloat16)
    h, w = put(rnd(T, K), run), put(rnd(E, K, seed=1, scale=K ** -0.5), run)
    ids, wt = ops.route(h, w, top)
    _, want = oracle.route(f64(h), f64(w), top)
    # as above
    assert (wt.cpu().double() - want).abs().max() < 6e-6
    s = oracle.sigmoid(f64(h) @ f64(w).T)
    assert (torch.gather(s, 1, ids.cpu().long()) - want).abs().max() < 6e-6


SHAPES = [(38, 11, 5), (64, 24, 7), (64, 64, 4), (192, 320, 6), (128, 200, 3)]


@pytest.mark.parametrize("run", RUNS)
@pytest.mark.parametrize("K,F,E", SHAPES)
class TestExperts:
    """Pairs per expert from one to hundreds: each form of the kernels."""

    def weights(self, run, K, F, E):
        return (put(rnd(E, F, K, seed=2, scale=K ** -0.5), run),
                put(rnd(E, K, F, seed=3, scale=F ** -0.5), run))

    def want(self, h, ids, wt, up, down):
        h, up, down, wt = f64(h), f64(up), f64(down), f64(wt)
        out = torch.zeros(ids.numel(), h.shape[1], dtype=F64)
        for p, e in enumerate(ids.flatten().tolist()):
            t = p // ids.shape[1]
            out[p] = oracle.expert(wt.flatten()[p] * h[t][None], up[e],
                                   down[e])[0]
        return out

    @pytest.mark.parametrize("T,top", [(1, 1), (3, 2), (50, 3), (130, 2),
                                       (400, 2)])
    def test_products(self, run, K, F, E, T, top):
        g = torch.Generator().manual_seed(T)
        up, down = self.weights(run, K, F, E)
        h = put(rnd(T, K), run)
        wt = (torch.rand(T, top, generator=g) * 0.9 + 0.05)
        ids = torch.stack([torch.randperm(E, generator=g)[:top]
                           for _ in range(T)]).int()
        out = ops.experts(h, ids.to(run[0]), wt.to(run[0]), up, down,
                          "relu_squared")
        want = self.want(h, ids, wt, up, down)
        close(out, want, run, f32=1e-5, bf16=2e-2)
        # the weight belongs to the input: on the output it would show
        bare = self.want(h, ids, torch.ones_like(wt), up, down)
        other = bare * wt.flatten()[:, None]
        assert (other - want).abs().max() > 0.1 * want.abs().max()

    def test_one_expert_takes_all(self, run, K, F, E):
        T = 150
        up, down = self.weights(run, K, F, E)
        h, wt = put(rnd(T, K), run), torch.full((T, 1), 0.7)
        ids = torch.full((T, 1), E - 1, dtype=torch.int32)
        ids[77] = 0
        out = ops.experts(h, ids.to(run[0]), wt.to(run[0]), up, down,
                          "relu_squared")
        close(out, self.want(h, ids, wt, up, down), run, f32=1e-5, bf16=2e-2)

    def test_rows_do_not_depend_on_the_batch(self, run, K, F, E):
        """A token alone and in a crowd."""
        up, down = self.weights(run, K, F, E)
        h = put(rnd(300, K), run)
        wt = torch.full((300, 2), 0.5, device=run[0])
        ids = torch.tensor([[1, 2], [0, 1], [2, 0]], dtype=torch.int32,
                           device=run[0]).repeat(100, 1)
        many = ops.experts(h, ids, wt, up, down, "relu_squared")
        for t in (0, 7, 299):
            one = ops.experts(h[t:t + 1].contiguous(),
                              ids[t:t + 1].contiguous(), wt[:1], up, down,
                              "relu_squared")
            close(one, f64(many[2 * t:2 * t + 2]), run, f32=1e-5, bf16=2e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("K,F", [(8, 8), (120, 136), (128, 64), (136, 1032), (520, 72),
                                 (1024, 256)])
@pytest.mark.parametrize("pairs", [1, 9, 12, 16, 17, 24, 33, 48])
def test_experts_of_few_pairs(K, F, pairs):
    """Each size of tiles: less than a step of K, remainders, channels past the end."""
    run, E = ("cuda", torch.bfloat16), 5
    up = put(rnd(E, F, K, seed=2, scale=K ** -0.5), run)
    down = put(rnd(E, K, F, seed=3, scale=F ** -0.5), run)
    g = torch.Generator().manual_seed(pairs)
    # all experts but one, unevenly: up to twice the mean number of pairs
    ids = torch.cat([torch.full((2 * pairs,), 4), torch.full((pairs,), 0),
                     torch.full((max(1, pairs - 3),), 2), torch.full((1,), 3)])
    ids = ids[torch.randperm(len(ids), generator=g)].int()[:, None]
    h = put(rnd(len(ids), K), run)
    wt = torch.rand(len(ids), 1, generator=g) * 0.9 + 0.05
    out = ops.experts(h, ids.cuda(), wt.cuda(), up, down, "relu_squared")
    want = TestExperts().want(h, ids, wt, up, down)
    # the inner rows and the results are rounded to 8 bits, 32-bit sums beside that
    close(out, want, run, bf16=2e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("K,F", [(128, 128), (192, 320), (576, 448)])
@pytest.mark.parametrize("counts", [(128, 129, 160), (192, 193, 0), (96, 145, 256),
                                    (321, 400, 449)])
def test_experts_of_many_pairs(K, F, counts):
    """Tiles of 128, 192 and 256 pairs: the ends of each, channels past the end."""
    run, E = ("cuda", torch.bfloat16), len(counts)
    up = put(rnd(E, F, K, seed=2, scale=K ** -0.5), run)
    down = put(rnd(E, K, F, seed=3, scale=F ** -0.5), run)
    g = torch.Generator().manual_seed(sum(counts))
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])
    ids = ids[torch.randperm(len(ids), generator=g)].int()[:, None]
    h = put(rnd(len(ids), K), run)
    wt = torch.rand(len(ids), 1, generator=g) * 0.9 + 0.05
    out = ops.experts(h, ids.cuda(), wt.cuda(), up, down, "relu_squared")
    want = TestExperts().want(h, ids, wt, up, down)
    # the inner rows and the results are rounded to 8 bits, 32-bit sums beside that
    close(out, want, run, bf16=2e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [8, 40, 90, 180])
def test_experts_of_a_row_whatever_others_chose(T):
    """Tiles of 16, 32 and 64 pairs: the first rows' bits, where the other rows have
    all experts and where they have few."""
    run, E, K, F = ("cuda", torch.bfloat16), 8, 1024, 776
    up = put(rnd(E, F, K, seed=2, scale=K ** -0.5), run)
    down = put(rnd(E, K, F, seed=3, scale=F ** -0.5), run)
    h, wt = put(rnd(T, K), run), torch.full((T, 2), 0.5, device="cuda")
    outs = []
    for low in (0, 4, 6):
        ids = torch.arange(T)[:, None] % (8 - low) + torch.tensor([low, low + 1])
        ids[:4] = torch.tensor([5, 7])
        out = ops.experts(h, (ids % 8).int().cuda(), wt, up, down, "relu_squared")
        outs.append(out[:8])       # four rows of two pairs
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@GPU
@pytest.mark.parametrize("D,V", [(64, 64), (128, 128), (192, 128), (64, 256)])
@pytest.mark.parametrize("bs", [1, 5, 64])
def test_prefill_in_other_pages(D, V, bs, monkeypatch):
    """Where keys and values lie changes no bit: block sizes that are powers of
    two and others, portions around tiles of 32 and 64 keys."""
    run, H, G = ("cuda:0", torch.bfloat16), 8, 2
    portions = [(0, 64), (31, 1), (200, 9), (63, 130), (0, 33)]
    seqs = [(n, prior, 0) for prior, n in portions]
    m, rows = meta(seqs, run)
    pos = torch.cat([torch.arange(a, a + n) for a, n in portions]).int()
    tiles = torch.tensor([(i, r) for i, (_, n) in enumerate(portions)
                          for r in range(0, n, 32)], dtype=torch.int32)
    proj = put(rnd(len(pos), H * D + G * (D + V), seed=3), run)
    outs = []
    for size in (16, bs):
        monkeypatch.setitem(globals(), "BS", size)
        cache, tables, _ = paged(run, G, D, V, [a + n for a, n in portions])
        out = put(torch.full((len(pos), H * V), 7.0), run)
        ops.grouped_prefill(proj, cache, pos.to(run[0]), rows, tables, 0, m,
                            tiles.to(run[0]), H, D, D ** -0.5, 0.0, out)
        outs.append(out)
    assert torch.equal(*outs)


@GPU
@pytest.mark.parametrize("D,bs", [(64, 8), (64, 4), (128, 4), (128, 2), (256, 2),
                                  (256, 1), (256, 128)])
def test_prefill_where_a_load_fits_a_page(D, bs, monkeypatch):
    """The smallest pages that hold the rows of a load whole, and smaller ones."""
    test_prefill_in_other_pages(D, D, bs, monkeypatch)



@GPU
def test_forms_agree_at_a_large_size():
    """The tiled products against the plain kernel."""
    dev, E, K, F, T, top = "cuda:0", 9, 512, 448, 1500, 3
    g = torch.Generator(device=dev).manual_seed(0)

    def normal(*shape, std=1.0):
        return torch.empty(shape, device=dev).normal_(
            0, std, generator=g).bfloat16()
    up, down = normal(E, F, K, std=K ** -0.5), normal(E, K, F, std=F ** -0.5)
    h = normal(T, K)
    ids, wt = ops.route(h, normal(E, K, std=K ** -0.5), top)
    a = ops.experts(h, ids, wt, up, down, "relu_squared")
    b = ops.experts(h, ids, wt, up, down, "relu_squared", plain=True)
    close(a, f64(b), ("", torch.bfloat16), bf16=1e-2)


@GPU
@pytest.mark.parametrize("K,F", [(128, 192), (192, 128), (320, 576)])
@pytest.mark.parametrize("act", ["relu_squared", "silu", "gelu_tanh"])
def test_tiles_at_their_edges(K, F, act):
    """Pairs of an expert around half and whole tiles, K of two steps and of
    more, channels that end inside a tile; against the plain kernel."""
    counts = [1, 128, 129, 0, 255, 256, 257, 384, 385, 512]
    dev, E, T = "cuda:0", len(counts), sum(counts)
    g = torch.Generator(device=dev).manual_seed(K + F)

    def normal(*shape, std=1.0):
        return torch.empty(shape, device=dev).normal_(
            0, std, generator=g).bfloat16()
    up, down = normal(E, F, K, std=K ** -0.5), normal(E, K, F, std=F ** -0.5)
    h = normal(T, K)
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])
    ids = ids[torch.randperm(T)].int().to(dev)[:, None].contiguous()
    wt = torch.rand(T, 1, device=dev, generator=g) * 0.9 + 0.05
    a = ops.experts(h, ids, wt, up, down, act)
    b = ops.experts(h, ids, wt, up, down, act, plain=True)
    close(a, f64(b), ("", torch.bfloat16), bf16=1e-2)


@GPU
@pytest.mark.parametrize("tile", [16, 32, 64, 256])
@pytest.mark.parametrize("share", [False, True])
@pytest.mark.parametrize("times", [-1, 0, 1, 2])
def test_order_of_tiles(tile, share, times):
    """Tiles more than half full first; by expert where they share weights: if
    some expert has several, of the large ones if every one has."""
    from llm_d_inference_scheduler_amd import _hip_layered as ext
    counts = [1, tile // 2, tile // 2 + 1, 0, tile - 1, tile, tile + 1]
    counts = counts[:6] + [0] * 70 if times < 0 else \
        [n + times * tile for n in counts]
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])
    ids = ids[torch.randperm(len(ids))].int()
    order, tiles = ext.sort_pairs(ids.cuda()[:, None], len(counts), tile,
                                  share)
    assert torch.equal(order.cpu().long(), ids.argsort(stable=True))
    cut, first = [], 0
    for e, n in enumerate(counts):
        cut += [[e, first + j, min(tile, n - j), 0] for j in range(0, n, tile)]
        first += n
    together = share and (max if tile < 256 else min)(counts) > tile
    if not together:
        cut.sort(key=lambda c: 2 * c[2] <= tile)
    ahead = sum(together or 2 * c[2] > tile for c in cut)
    assert tiles[0, :2].tolist() == [len(cut), ahead]
    assert tiles[1:1 + len(cut)].tolist() == cut


@GPU
def test_tiles_that_share_weights():
    """Experts whose weights do not stay in a cache, several tiles each."""
    dev, E, K, F = "cuda:0", 5, 8192, 8192
    counts = [257, 300, 384, 400, 512]
    g = torch.Generator(device=dev).manual_seed(0)

    def normal(*shape, std=1.0):
        return torch.empty(shape, device=dev).normal_(
            0, std, generator=g).bfloat16()
    up, down = normal(E, F, K, std=K ** -0.5), normal(E, K, F, std=F ** -0.5)
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(counts)])
    ids = ids[torch.randperm(len(ids))].int().to(dev)[:, None].contiguous()
    h, wt = normal(len(ids), K), torch.ones(len(ids), 1, device=dev)
    got = ops.experts(h, ids, wt, up, down, "silu")
    for e in range(E):
        rows = (ids[:, 0] == e).nonzero()[:, 0]
        inner = torch.nn.functional.silu(h[rows].float() @ up[e].float().t())
        close(got[rows], f64(inner @ down[e].float().t()),
              ("", torch.bfloat16), bf16=1e-2)
