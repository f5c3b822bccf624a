"""plan_step's arrays against the same arrays made entry by entry."""
import random

import numpy as np
import pytest

from swiftllm_amd.worker.batch_plan import StepEntry, StepPlan, plan_step, plan_tokens


def _by_entry(entries):
    out = {name: [] for name in StepPlan.SEGMENTS}
    at = tiles = chunks = 0
    for e in entries:
        n = len(e.tokens)
        out["input_ids"] += list(e.tokens)
        out["tok_pos"] += range(e.start, e.start + n)
        out["tok_seq"] += [e.seq_id] * n
        out["tok_start"] += [e.start] * n
        out["tok_state"] += [0] * n
        out["want_rows"] += [at + w for w in e.want]
        out["seq_row0"].append(at)
        out["seq_cnt"].append(n)
        out["seq_tile0"].append(tiles)
        out["seq_chunk0"].append(chunks)
        for what, size in (("tile", StepPlan.TILE), ("chunk", StepPlan.CHUNK)):
            out[what + "_row0"] += range(at, at + n, size)
            out[what + "_cnt"] += [min(size, n - i) for i in range(0, n, size)]
        at, tiles, chunks = at + n, tiles + -(-n // StepPlan.TILE), chunks + -(-n // StepPlan.CHUNK)
    return out


@pytest.mark.parametrize("lens", [[], [1], [1, 1, 1], [2, 1], [16, 17, 15, 1], [31, 32, 33, 64, 100, 1, 1]])
def test_arrays(lens):
    rng = random.Random(len(lens))
    entries = [StepEntry(3 * i + 1, [rng.randrange(50) for _ in range(n)], rng.choice([0, 7, 130]), tuple(rng.sample(range(n), rng.randint(0, min(2, n)))))
               for i, n in enumerate(lens)]
    entries = [StepEntry(e.seq_id, np.asarray(e.tokens), e.start, e.want) if rng.random() < 0.3 else e for e in entries]
    plan = plan_step(entries, 50, 300)
    for name, want in _by_entry(entries).items():
        got = getattr(plan, name)
        assert got.dtype == np.int32 and got.tolist() == want, name
    assert plan.num_tokens == sum(lens) and plan.num_seqs == len(lens)
    assert plan.seq_ids_list == [e.seq_id for e in entries] and plan.target_lens_list == [e.start + len(e.tokens) for e in entries]


def test_the_first_bad_entry_is_reported():
    good = StepEntry(1, [3, 4], 0, (1,))
    for bad, kind, text in ((StepEntry(2, [], 0), ValueError, "brings no tokens"), (StepEntry(2, [1], -1), ValueError, "negative start"),
                            (StepEntry(2, [1, 2], 9), RuntimeError, "would reach position 10"), (StepEntry(1, [5], 0), ValueError, "appears twice"),
                            (StepEntry(2, [50], 0), ValueError, r"must be in \[0, 50\)"), (StepEntry(2, [-1, 3], 0), ValueError, "must be in"),
                            (StepEntry(2, [1], 0, (1,)), ValueError, "wanted offset 1"), (StepEntry(2, [1], 0, (-1,)), ValueError, "wanted offset -1")):
        with pytest.raises(kind, match=text):
            plan_step([good, bad, StepEntry(5, [], -1)], 50, 10)


@pytest.mark.parametrize("bad,kind,text", [
    (StepEntry(2, [1], 1 << 40), RuntimeError, "would reach position"), (StepEntry(2, [1], -(1 << 40)), ValueError, "negative start"),
    (StepEntry(2, [1 << 63], -1), ValueError, "negative start"), (StepEntry(2, [1 << 63], 0), OverflowError, ""),
    (StepEntry(1 << 40, [1], 0, (3,)), OverflowError, ""), (StepEntry(2, [1 << 40], 0), ValueError, r"must be in \[0, 50\)")])
def test_values_beyond_32_bits(bad, kind, text):
    """What no int32 holds is refused with the error that the entry's other faults get, the first bad entry's."""
    with pytest.raises(kind, match=text):
        plan_step([StepEntry(1, [3, 4], 0, (1,)), bad, StepEntry(5, [], -1)], 50, 10)


def test_positions_end_with_32_bits():
    """Without a position table the last position is 2^31 - 1: a portion that passes it is refused, not wrapped round."""
    assert plan_step([StepEntry(1, [3, 4], (1 << 31) - 2)]).tok_pos.tolist() == [(1 << 31) - 2, (1 << 31) - 1]
    for start in ((1 << 31) - 1, 1 << 31):
        with pytest.raises(OverflowError):
            plan_step([StepEntry(1, [3, 4], start)])


def test_span_order_takes_runs_of_four_from_the_highest_positions():
    """A permutation; runs of four chunks of a portion stay together, last chunk first; runs come in descending position; small steps have
    none."""
    assert plan_step([StepEntry(0, [1] * 2048, 0)]).span_order() is None        # (64 chunks)
    parts = [(0, 0, 1000), (1, 77, 1), (2, 40, 900), (3, 0, 31), (4, 5, 385)]
    plan = plan_step([StepEntry(i, [1] * n, a) for i, a, n in parts])
    order = plan.span_order()
    assert order.dtype == np.int32 and sorted(order) == list(range(plan.chunk_row0.size))
    runs, at = [], 0
    for i, a, n in parts:
        chunks = -(-n // 32)
        runs += [(a + 128 * k, i, [at + c for c in range(min(4 * k + 4, chunks) - 1, 4 * k - 1, -1)]) for k in range(-(-chunks // 4))]
        at += chunks
    runs.sort(key=lambda r: (-r[0], -r[1]))
    assert order.tolist() == [c for r in runs for c in r[2]]


@pytest.mark.parametrize("parts,ordered", [([(0, 2000)] + [(800, 1)] * 30, False), ([(0, 4096)], False), ([(0, 4097)], True),
                                           ([(0, 333)] * 12, True), ([(0, 333)] * 11, False), ([(5, 1)] * 200, False)])
def test_small_steps_go_without_an_order(parts, ordered):
    """Up to 128 spans (and in steps of one token each) the order costs the host more than it gives the launches."""
    plan = plan_step([StepEntry(i, [1] * n, a) for i, (a, n) in enumerate(parts)])
    order = plan.upload_order()
    assert (order is not None) == ordered
    assert order is None or order.tolist() == plan.span_order().tolist()


@pytest.mark.parametrize("n", [1, 2, 3, 33, 65])
def test_plan_of_one_token_each(n):
    """plan_tokens is plan_step of the same entries, array for array, and gives none where plan_step refuses."""
    rng = random.Random(n)
    toks, ids, starts = [rng.randrange(50) for _ in range(n)], rng.sample(range(100), n), [rng.randrange(300) for _ in range(n)]
    for given in (toks, [np.int64(t) for t in toks]):
        plan = plan_tokens(given, ids, starts, 50, 300)
        want = plan_step([StepEntry(i, [t], a, (0,)) for i, t, a in zip(ids, toks, starts)], 50, 300)
        for name in StepPlan.SEGMENTS:
            got = getattr(plan, name)
            assert got.dtype == np.int32 and got.tolist() == getattr(want, name).tolist(), name
        assert (plan.num_tokens, plan.num_seqs, plan.seq_ids_list, plan.target_lens_list) == (n, n, want.seq_ids_list, want.target_lens_list)
        assert plan.span_order() is None
    at = rng.randrange(n)
    for which, bad in ((0, 50), (0, -1), (0, 1 << 63), (1, 1 << 40), (2, -1), (2, 300), (2, 1 << 40)):
        lists = [list(toks), list(ids), list(starts)]
        lists[which][at] = bad
        assert plan_tokens(*lists, 50, 300) is None
        with pytest.raises((ValueError, RuntimeError, OverflowError)):
            plan_step([StepEntry(i, [t], a, (0,)) for t, i, a in zip(*lists)], 50, 300)
    if n > 1:
        assert plan_tokens(toks, ids[:-1] + ids[:1], starts, 50, 300) is None
    assert plan_tokens([], [], [], 50, 300) is None


@pytest.mark.parametrize("window", [0, 48])
def test_latent_expansion_covers_what_its_portions_see(window):
    """Every page that a query of an expanded portion sees is expanded once, under the number that the attention's table gives it; what is
    left keeps its chunks and tiles."""
    from swiftllm_amd.worker.batch_plan import LatentExpansion
    rng = random.Random(window)
    spec = LatentExpansion(128, 64, 128, 512, window, 4096)
    for _ in range(60):
        parts = [(s, rng.choice((0, 0, rng.randint(0, 300))), rng.choice((1, 17, rng.randint(16, 260)))) for s in rng.sample(range(40), rng.randint(1, 6))]
        plan = plan_step([StepEntry(s, [1] * n, a, ()) for s, a, n in parts])
        ex = plan.latent_expansion(spec)
        pays = spec.pays(np.array([a for _, a, _ in parts]), np.array([n for _, _, n in parts])).tolist()
        k = (pays + [False]).index(False)
        if k == 0:
            assert ex is None
            continue
        A = ex.arrays
        assert sum((v.size + 3) // 4 * 4 for v in A.values()) <= spec.most_ints(plan.num_tokens, len(parts), max(-(-(a + n) // 16) for _, a, n in parts))
        assert ex.seqs == k and ex.rows == sum(n for _, _, n in parts[:k])
        made = {int(d): (int(r), int(p)) for r, p, d in zip(A["ex_page_row"], A["ex_page_no"], A["ex_page_dst"])}
        assert len(made) == A["ex_page_dst"].size and max(made) < ex.pages == A["ex_table"].size
        row, first = 0, []
        for s, a, n in parts[:k]:
            rows = A["ex_tok_row"][row:row + n]
            assert (rows == rows[0]).all()
            first.append(int(rows[0]))
            for page in range((max(a - window + 1, 0) if window else 0) // 16, (a + n - 1) // 16 + 1):
                assert made.pop(int(A["ex_table"][rows[0] + page])) == (s, page)
            row += n
        assert not made and len(set(first)) == k
        if k < len(parts):
            assert np.array_equal(A["ex_rest_chunk_row0"] + row, plan.chunk_row0[ex.chunks:]) and plan.chunk_row0[ex.chunks] == row
            assert np.array_equal(A["ex_rest_tile_row0"] + row, plan.tile_row0[ex.tiles:]) and plan.tile_row0[ex.tiles] == row
        order = plan.upload_order()
        if order is not None:
            assert sorted(A["ex_order"]) == list(range(ex.chunks))


@pytest.mark.parametrize("tokens,beside,expanded", [(100, 0, True), (63, 3, False), (64, 3, True), (200, 1, True), (16, 30, False)])
def test_latent_expansion_beside_folded_portions(tokens, beside, expanded):
    """Beside portions that stay folded a step expands from min_beside tokens on, alone always."""
    from swiftllm_amd.worker.batch_plan import LatentExpansion
    entries = [StepEntry(0, [1] * (tokens // 2), 0, ()), StepEntry(1, [1] * (tokens - tokens // 2), 0, ())] if tokens >= 32 else [StepEntry(0, [1] * tokens, 0, ())]
    plan = plan_step(entries + [StepEntry(9 + i, [1], 20, (0,)) for i in range(beside)])
    ex = plan.latent_expansion(LatentExpansion(128, 64, 128, 512, 0, 4096, 64))
    assert (ex is not None and ex.rows == tokens) == expanded and (expanded or ex is None)


@pytest.mark.parametrize("dim,rot,vdim,rank,start,count,pays", [(128, 64, 128, 512, 0, 16, True), (128, 64, 128, 512, 1000, 64, True), (128, 64, 128, 512, 3000, 17, False),
                                                                (64, 64, 128, 128, 0, 2000, False), (64, 64, 128, 128, 0, 100, False),
                                                                (128, 64, 128, 256, 0, 2000, True), (128, 64, 128, 256, 3000, 128, False)])
def test_latent_expansion_by_the_rank(dim, rot, vdim, rank, start, count, pays):
    """The heads' own keys have to be a good deal narrower than folded rows: they are staged for one head alone."""
    from swiftllm_amd.worker.batch_plan import LatentExpansion
    assert LatentExpansion(dim, rot, vdim, rank, 0, 4096).pays(np.array([start]), np.array([count])).tolist() == [pays]
