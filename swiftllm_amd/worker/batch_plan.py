"""Host-side batch planning: everything `LlamaModel.forward` derives from its Python-list arguments
before touching the device. Pure numpy — unit-tested on CPU against the reference's arithmetic.

Reference: swiftllm/worker/model.py:268-324 (flattening, sequence lengths, start offsets, position
indices, the seq_block_size heuristic) and post_layer.py:24-29 (last-token indices).
"""
import dataclasses
import itertools
from typing import List, Sequence

import numpy as np


def select_seq_block_size(decoding_seq_lens: Sequence[int], num_kv_heads: int,
                          num_slots: int = 256, max_splits: int = 128) -> int:
    """Split-K width (tokens) of flash-decoding, sized for MI355X.

    The reference halves 2048 until `KVH * sum(len) / width >= 1024` programs exist (model.py:305-324:
    "1024 because ~128 SMs", one 1-warp program per q-head). Our phase-1 workgroup is 8 waves serving
    a whole kv-head group, one per CU, so the right launch is ~`num_slots` (= CU count, 256)
    workgroups in whole rounds, each with as many KV blocks as possible:

        width = KVH * sum(len) / num_slots        (tokens per workgroup for one full round)

    rounded up to 64 tokens. When that width already covers the longest sequence there is a single
    sequence block per sequence — phase 1 writes the output directly and phase 2 is never launched —
    and the width is rounded up to 256 so it (and a captured hipGraph) stays valid while the
    sequences grow. The width is a free internal choice: results are invariant up to fp32
    reassociation, which tests/test_gpu_kernels.py checks.
    """
    if len(decoding_seq_lens) == 0:
        return 2048
    total = sum(-(-n // 64) * 64 for n in decoding_seq_lens)
    longest = max(decoding_seq_lens)
    size = max(64, -(-(num_kv_heads * total) // (num_slots * 64)) * 64)
    if size >= longest:
        size = -(-size // 256) * 256
    while -(-longest // size) > max_splits:
        size *= 2
    return size


def decode_attention_waves(num_seqs: int, longest: int, num_kv_heads: int, seq_block_size: int, num_slots: int = 256) -> int:
    """Waves of a workgroup of the slab-fed decode attention (csrc/paged_attn.hip, launch_phase1): four where the sequence blocks are short
    or the launch of these sequences as they are has more workgroups than there are CUs; eight otherwise. `num_seqs` real ones: neither the
    inert sequences of a batch rounded up to its replay bucket nor its splits rounded up to a power of two count, so that they change the
    order of nobody's sums. Workgroups past a sequence's end do count: 36 batches of 2 to 15 sequences with the longest at 2.2k to 15k,
    whose 240 to 264 working ones are in a grid of 304 to 768, all take 10 to 33 % less with four waves (5 of up to 4.7k: 22.7 and
    27.4 us; 8 kv heads of 128); 4 of 4000 in a grid of 256 take 20.2 and 17.6 us."""
    if seq_block_size < 512:
        return 4
    return 4 if num_kv_heads * num_seqs * -(-longest // seq_block_size) > num_slots else 8


@dataclasses.dataclass
class BatchPlan:
    batch_size: int
    num_tokens: int
    num_prefill_seqs: int
    num_prefill_tokens: int
    max_prefill_len: int
    num_decoding_seqs: int
    max_decoding_len: int
    seq_block_size: int
    num_seq_blocks: int
    seq_lengths_list: List[int]
    # int32 arrays
    input_ids: np.ndarray               # [T]
    seq_ids: np.ndarray                 # [B]
    seq_lengths: np.ndarray             # [B]
    prefill_seq_lens: np.ndarray        # [Bp]
    prefill_start_locs_with_end: np.ndarray  # [Bp + 1]
    decoding_seq_lens: np.ndarray       # [Bd]
    position_indices: np.ndarray        # [T]
    last_token_indices: np.ndarray      # [B]
    # sequences of the caller's batch; batch_size - num_real_seqs trailing rows are inert padding (length 0) that rounds a
    # pure-decode batch up to its hipGraph bucket (worker/model.py: _decode_batch_bucket). -1: not set = batch_size
    num_real_seqs: int = -1

    @property
    def real_seqs(self) -> int:
        return self.num_real_seqs if self.num_real_seqs >= 0 else self.batch_size

    SEGMENTS = ("input_ids", "seq_ids", "seq_lengths", "prefill_seq_lens",
                "prefill_start_locs_with_end", "decoding_seq_lens", "position_indices",
                "last_token_indices")

    def packed_layout(self):
        """(name, offset, size) of every array inside one int32 buffer; offsets are multiples of 4
        elements (16 bytes). The layout depends only on (T, B, Bp), so a replayed hipGraph of a
        pure-decode batch of size B always finds its metadata at the same addresses."""
        out, off = [], 0
        for name in self.SEGMENTS:
            n = getattr(self, name).size
            out.append((name, off, n))
            off += (n + 3) // 4 * 4
        return out, off

    def pack_into(self, buf: np.ndarray) -> int:
        layout, total = self.packed_layout()
        for name, off, n in layout:
            buf[off:off + n] = getattr(self, name)
        return total


def plan_batch(input_ids_list: Sequence[Sequence[int]], seq_ids_list: Sequence[int],
               decoding_seq_lens_list: Sequence[int], num_kv_heads: int,
               num_slots: int = 256) -> BatchPlan:
    """Prefill sequences come first in all three lists (reference model.py:268-270); a decoding
    sequence contributes exactly one token and its length INCLUDES that token."""
    batch_size = len(input_ids_list)
    num_decoding = len(decoding_seq_lens_list)
    num_prefill = batch_size - num_decoding
    if num_prefill < 0 or len(seq_ids_list) != batch_size:
        raise ValueError("inconsistent batch: need len(seq_ids) == len(input_ids) >= len(decoding_seq_lens)")
    prefill_lens = [len(ids) for ids in input_ids_list[:num_prefill]]
    flat = np.fromiter(itertools.chain.from_iterable(input_ids_list), dtype=np.int32)
    num_tokens = flat.size
    num_prefill_tokens = sum(prefill_lens)
    if num_tokens - num_prefill_tokens != num_decoding:
        raise ValueError("every decoding sequence must contribute exactly one token")
    pl = np.asarray(prefill_lens, dtype=np.int32)
    dl = np.asarray(decoding_seq_lens_list, dtype=np.int32)
    starts_with_end = np.zeros(num_prefill + 1, dtype=np.int32)
    np.cumsum(pl, out=starts_with_end[1:])
    pos = np.empty(num_tokens, dtype=np.int32)
    if num_prefill_tokens:
        # 0..len-1 for every prefill sequence: global arange minus each token's sequence start
        pos[:num_prefill_tokens] = (np.arange(num_prefill_tokens, dtype=np.int32)
                                    - np.repeat(starts_with_end[:-1], pl))
    pos[num_prefill_tokens:] = dl - 1
    last = np.concatenate((starts_with_end[1:] - 1,
                           np.arange(num_prefill_tokens, num_tokens, dtype=np.int32))).astype(np.int32)
    sbs = select_seq_block_size(decoding_seq_lens_list, num_kv_heads, num_slots)
    max_dec = max(decoding_seq_lens_list) if num_decoding else 0
    seq_lengths_list = prefill_lens + list(decoding_seq_lens_list)
    return BatchPlan(
        batch_size=batch_size, num_tokens=num_tokens, num_prefill_seqs=num_prefill,
        num_prefill_tokens=num_prefill_tokens,
        max_prefill_len=max(prefill_lens) if prefill_lens else 0,
        num_decoding_seqs=num_decoding, max_decoding_len=max_dec, seq_block_size=sbs,
        num_seq_blocks=(max_dec + sbs - 1) // sbs, seq_lengths_list=seq_lengths_list,
        input_ids=flat, seq_ids=np.asarray(seq_ids_list, dtype=np.int32),
        seq_lengths=np.asarray(seq_lengths_list, dtype=np.int32), prefill_seq_lens=pl,
        prefill_start_locs_with_end=starts_with_end, decoding_seq_lens=dl, position_indices=pos,
        last_token_indices=last)


# ---- token-level steps: prompt portions and decoded tokens in one batch ----------------------------------------------------
@dataclasses.dataclass
class StepEntry:
    """The tokens one sequence brings to a step: `tokens` continue the sequence at position `start` (0 for a new sequence;
    a decoded token is a portion of length one). `want`: offsets inside `tokens` whose logits the caller asks for."""
    seq_id: int
    tokens: Sequence[int]
    start: int
    want: Sequence[int] = ()


class LatentExpansion:
    """What decides whether the latent attention of a portion runs on the heads' own keys and values, expanded from the cached rows
    (csrc/latent_expand.hip), or on queries folded through the key up-projection: the matrix steps of both, by the sizes of the layers.
    window: of the layers' the largest, 0 if one sees every key; max_pages: pages that the expansion may take; min_beside: tokens it takes
    beside portions that stay folded."""
    MIN_TOKENS = 16

    def __init__(self, dim: int, rot_dim: int, vdim: int, rank: int, window: int, max_pages: int, min_beside: int = 0):
        self.window, self.max_pages, self.min_beside = window, max_pages, min_beside
        # tenths of a column: what a visible (query, key) pair costs more when folded (values count twice; a column of the heads' own keys, which
        # a workgroup stages for one head alone, 1.3 of one for all), and what expanding one more key costs
        self.pair_gain = 10 * (3 * rank + rot_dim) - 13 * (dim + rot_dim + 2 * vdim)
        self.key_cost = 10 * (dim + vdim) * rank

    def pays(self, start: np.ndarray, count: np.ndarray) -> np.ndarray:
        """By portion: its own keys take as long to expand as its queries to fold; keys before it are extra. A column of the expansion takes
        half as long as one of attention. Measured, us from the projection to the heads' results, 8 heads of 128 + 64 over rank 512 in a window
        of 1024, folded and expanded: 16 tokens 34.9, 21.4; 11 x 333 94.7, 57.0; 4 x 2000 276, 165; 64 behind 1000 50.2, 33.1; 8 x 64 behind
        1000 67.6, 66.2; 8 x 128 98.5, 69.4. 16 heads, no window: 4 x 2000 566, 350; 8 x 64 behind 1000 97.8, 88.6; 8 x 128 behind 3000 277, 269.
        By rank, no window: 40 heads of 64 + 64 and 128 over 128 (448 columns against 384, never expanded) 100 tokens 29, 24; 500 49, 46; 11 x 333 150, 164;
        2000 181, 277; 4 x 500 behind 500 154, 248; 8 heads 2000 66, 62; 8 heads of 128 + 64 over 256 4 x 128 behind 3000 71, 74."""
        before, seen = start, count * (2 * start + count + 1) // 2      # (seen: pairs)
        if self.window > 0:
            before, seen = np.minimum(start, self.window - 1), np.minimum(seen, count * self.window)
        return (count >= self.MIN_TOKENS) & (2 * seen * self.pair_gain > before * self.key_cost)

    def most_ints(self, tokens: int, portions: int, pages: int) -> int:
        """Ints that a step's orders and the arrays of its expansion (ExpandedPortions, each on 16 bytes) take at most: so many tokens, portions,
        and pages of a portion."""
        pages = min(pages * portions, self.max_pages)
        chunks, tiles = tokens // StepPlan.CHUNK + portions, tokens // StepPlan.TILE + portions
        return 4 * pages + tokens + 3 * chunks + tiles + 9 * 4


class ExpandedPortions:
    """The first `seqs` portions of a step (`rows` tokens, `chunks` chunks, `tiles` tiles) on `pages` expanded pages. arrays: int32, for the
    device: the pages to expand (block-table row, page, its number), ex_tok_row: what ex_table's entry of a token's page is the page's
    number less (attention finds page i of a portion at ex_table[ex_tok_row + i]), ex_order: the order of the portions' spans, and the
    first rows of the other portions' chunks and tiles counted from theirs."""
    __slots__ = ("seqs", "rows", "chunks", "tiles", "pages", "arrays")

    def __init__(self, seqs, rows, chunks, tiles, pages, arrays):
        self.seqs, self.rows, self.chunks, self.tiles, self.pages, self.arrays = seqs, rows, chunks, tiles, pages, arrays


@dataclasses.dataclass
class StepPlan:
    """Flat per-token metadata of a step. Kernels that serve portions and decoded tokens alike need nothing else: a token's
    block-table row, its position, and (for the output) which rows are asked for."""
    num_tokens: int
    num_seqs: int
    seq_ids_list: List[int]
    target_lens_list: List[int]         # length of every sequence after the step (what the block allocator must cover)
    input_ids: np.ndarray               # [T] int32
    tok_pos: np.ndarray                 # [T] int32 position of each token in its sequence
    tok_seq: np.ndarray                 # [T] int32 block-table row of each token
    want_rows: np.ndarray               # [R] int32 rows (into the T tokens) whose logits are produced
    # tiles of up to TILE consecutive tokens of one sequence (the matrix-core attention's unit of work)
    tile_row0: np.ndarray = None        # [NT] int32 first token row of each tile
    tile_cnt: np.ndarray = None         # [NT] int32 tokens in it
    # the portions themselves (what recurrent layers walk token by token) and, per token, where its portion starts
    seq_row0: np.ndarray = None         # [S] int32 first token row of each sequence's portion
    seq_cnt: np.ndarray = None          # [S] int32 tokens in it
    tok_start: np.ndarray = None        # [T] int32 position of the first token of the token's portion
    # [T] int32 state slot * 2 + tail parity of the token's sequence; zeros until a worker with per-sequence state fills it
    tok_state: np.ndarray = None
    # the portions cut into runs of up to CHUNK tokens (what a recurrence that is linear in its state evaluates in parallel), and
    # the first of each sequence's
    chunk_row0: np.ndarray = None       # [NC] int32 first token row of each chunk
    chunk_cnt: np.ndarray = None        # [NC] int32 tokens in it
    seq_chunk0: np.ndarray = None       # [S] int32
    seq_tile0: np.ndarray = None        # [S] int32 the first tile of each sequence

    TILE = 16
    CHUNK = 32
    SEGMENTS = ("input_ids", "tok_pos", "tok_seq", "want_rows", "tile_row0", "tile_cnt", "seq_row0", "seq_cnt", "tok_start",
                "tok_state", "chunk_row0", "chunk_cnt", "seq_chunk0", "seq_tile0")

    def span_order(self):
        """The chunks in the order in which attention takes them up, int32: runs of four of a portion (128 tokens, nearly the same
        keys) together, the runs at the highest positions first. None for steps so small that all are taken up at once, and for steps of
        one token each, whose attention reads no spans (128 decoded tokens: the order took 20 us of the host, with the device idle)."""
        n = self.chunk_row0.size
        if n <= 64 or n == self.num_tokens:
            return None
        portion = np.repeat(np.arange(self.num_seqs), np.diff(self.seq_chunk0, append=n))
        first = self.tok_pos[self.chunk_row0] - ((np.arange(n) - self.seq_chunk0[portion]) & 3) * self.CHUNK      # position of the run
        key = first.astype(np.int64) * self.num_seqs + portion
        return (n - 1 - np.argsort(-key[::-1], kind="stable")).astype(np.int32)

    # Steps of up to so many spans go without: making and packing the order takes a step 25 us of the host (10 in a loop of nothing else), with
    # the device idle, and it gives a launch at most 3 us there (8 or 4 heads of 128 over 2 or 4, 66 to 128 spans; 16 heads over 4 up to 7, 8
    # latent heads over one none), against 1 to 22 us at 220 and more. A step of 2030 tokens (94 spans, three such launches) 1322 -> 1315 us
    # without it, one of 3663 (121) 3010 -> 2995.
    ORDER_MIN_SPANS = 128

    def upload_order(self):
        """span_order where it pays, or None."""
        return self.span_order() if self.chunk_row0.size > self.ORDER_MIN_SPANS else None

    def latent_expansion(self, spec: "LatentExpansion"):
        """The portions at the head of the step whose latent attention runs on expanded pages (spec.pays says which gain by it): ->
        ExpandedPortions, or None where there is none."""
        count = np.asarray(self.seq_cnt, dtype=np.int64)
        if count.size == 0 or count[0] < LatentExpansion.MIN_TOKENS:
            return None
        if self.num_tokens < spec.min_beside and count.min() < LatentExpansion.MIN_TOKENS:      # (one stays folded, the others are too few)
            return None
        start = self.tok_pos[self.seq_row0].astype(np.int64)
        first = np.maximum(start - spec.window + 1, 0) // 16 if spec.window > 0 else np.zeros_like(start)    # first page with a visible key
        pages = -(-(start + count) // 16)
        # a portion's pages are numbered from `at` on, those before the first visible one too: `at` tells portions apart
        at = np.cumsum(pages) - pages
        ok = spec.pays(start, count) & (at + pages <= spec.max_pages)
        k = ok.size if ok.all() else int(np.argmin(ok))
        if k == 0:
            return None
        rest = k < ok.size
        row0, chunk0, tile0 = ((int(self.seq_row0[k]), int(self.seq_chunk0[k]), int(self.seq_tile0[k])) if rest else
                               (self.num_tokens, self.chunk_row0.size, self.tile_row0.size))
        if rest and row0 < spec.min_beside:
            return None
        first, pages, at, count = first[:k], pages[:k], at[:k], count[:k]
        each = pages - first
        page_no = np.arange(int(each.sum())) - np.repeat(np.cumsum(each) - each - first, each)
        i32, numbers = np.int32, int(at[-1] + pages[-1])
        arrays = {"ex_page_row": np.repeat(self.tok_seq[self.seq_row0[:k]], each), "ex_page_no": page_no.astype(i32),
                  "ex_page_dst": (page_no + np.repeat(at, each)).astype(i32), "ex_tok_row": np.repeat(at, count).astype(i32),
                  "ex_table": np.arange(numbers, dtype=i32)}
        order = self.upload_order()
        if order is not None:
            arrays["ex_order"] = order[order < chunk0]
        if rest:
            arrays["ex_rest_chunk_row0"] = self.chunk_row0[chunk0:] - i32(row0)
            arrays["ex_rest_tile_row0"] = self.tile_row0[tile0:] - i32(row0)
        return ExpandedPortions(k, row0, chunk0, tile0, numbers, arrays)

    def packed_layout(self):
        out, off = [], 0
        for name in self.SEGMENTS:
            n = getattr(self, name).size
            out.append((name, off, n))
            off += (n + 3) // 4 * 4
        return out, off

    def pack_into(self, buf: np.ndarray) -> int:
        layout, total = self.packed_layout()
        for name, off, n in layout:
            buf[off:off + n] = getattr(self, name)
        return total


def _check_entries(entries: Sequence[StepEntry], vocab_size, max_positions):
    """Raises what is wrong with the first entry that has anything wrong."""
    seen = set()
    for e in entries:
        n = len(e.tokens)
        if n == 0:
            raise ValueError(f"sequence {e.seq_id} brings no tokens to the step")
        if e.start < 0:
            raise ValueError(f"sequence {e.seq_id}: negative start {e.start}")
        if max_positions is not None and e.start + n > max_positions:
            raise RuntimeError(f"sequence {e.seq_id} would reach position {e.start + n - 1}, the model has "
                               f"{max_positions} positions")
        if e.seq_id in seen:
            raise ValueError(f"sequence {e.seq_id} appears twice in one step")
        toks = np.asarray(e.tokens, dtype=np.int64)
        if vocab_size is not None and (toks.min() < 0 or toks.max() >= vocab_size):
            raise ValueError(f"sequence {e.seq_id}: token ids must be in [0, {vocab_size})")
        np.arange(e.start, e.start + n, dtype=np.int32), np.full(n, e.seq_id, dtype=np.int32)      # (OverflowError: not in 32 bits)
        for w in e.want:
            if not 0 <= w < n:
                raise ValueError(f"sequence {e.seq_id}: wanted offset {w} outside its {n} tokens")
        seen.add(e.seq_id)


def plan_step(entries: Sequence[StepEntry], vocab_size: int = None, max_positions: int = None) -> StepPlan:
    """Flatten the entries in order. Checked here, on the host, so that nothing out of range reaches a kernel: token ids
    against the vocabulary, positions against the position table (and 32 bits), one entry per sequence.
    The device waits for this between two decode steps, so the arrays are made whole, not entry by entry: 32 decoded tokens
    480 -> 50 us, 3 70 -> 24 us. Values that no array holds are reported like the others: the first bad entry's."""
    try:
        return _plan_whole(entries, vocab_size, max_positions)
    except (OverflowError, ValueError, TypeError):
        _check_entries(entries, vocab_size, max_positions)
        raise


def plan_tokens(tokens: Sequence[int], seq_ids: Sequence[int], starts: Sequence[int], vocab_size: int = None, max_positions: int = None):
    """plan_step of one wanted token for each sequence (StepEntry(seq_id, [token], start, (0,)) in order), or None where anything is out of
    range: plan_step says what. A decode step waits for this with an idle device; 32 sequences 58 -> 15 us with the entries that it does
    without, 3 sequences 23 -> 10."""
    i32, n = np.int32, len(seq_ids)
    try:
        toks = np.asarray(tokens, dtype=np.int64)
        ids, first, known = [int(s) for s in seq_ids], [int(a) for a in starts], toks.tolist()
        targets = [a + 1 for a in first]
        if not (n and toks.shape == (n,) and len(first) == n and min(first) >= 0 and len(set(ids)) == n
                and max(targets) <= (1 << 31 if max_positions is None else min(max_positions, 1 << 31))
                and (vocab_size is None or (min(known) >= 0 and max(known) < vocab_size))):
            return None
        pos, seq, toks = np.asarray(first, dtype=i32), np.asarray(ids, dtype=i32), toks.astype(i32)
    except (OverflowError, ValueError, TypeError):
        return None
    rows, ones = np.arange(n, dtype=i32), np.ones(n, dtype=i32)
    return StepPlan(num_tokens=n, num_seqs=n, seq_ids_list=ids, target_lens_list=targets, input_ids=toks, tok_pos=pos, tok_seq=seq,
                    want_rows=rows, tile_row0=rows, tile_cnt=ones, seq_row0=rows, seq_cnt=ones, tok_start=pos,
                    tok_state=np.zeros(n, dtype=i32), chunk_row0=rows, chunk_cnt=ones, seq_chunk0=rows, seq_tile0=rows)


def _plan_whole(entries: Sequence[StepEntry], vocab_size, max_positions) -> StepPlan:
    i32 = np.int32
    seq_ids = [int(e.seq_id) for e in entries]
    lens = [len(e.tokens) for e in entries]
    starts_list = [int(e.start) for e in entries]
    targets = [a + n for a, n in zip(starts_list, lens)]
    base = sum(lens)
    counts, starts = np.asarray(lens, dtype=i32), np.asarray(starts_list, dtype=i32)
    row0 = (np.cumsum(counts) - counts).astype(i32)
    if base == len(lens):       # one token each
        toks = np.asarray([t for e in entries for t in e.tokens], dtype=np.int64)
    else:
        toks = np.concatenate([np.asarray(e.tokens, dtype=np.int64) for e in entries])
    want, wants_ok, at = [], True, 0
    for e, n in zip(entries, lens):
        for w in e.want:
            wants_ok = wants_ok and 0 <= w < n
            want.append(at + w)
        at += n
    if entries and not (wants_ok and min(lens) > 0 and min(starts_list) >= 0 and len(set(seq_ids)) == len(seq_ids)
                        and max(targets) <= (1 << 31 if max_positions is None else min(max_positions, 1 << 31))
                        and (vocab_size is None or (toks.min() >= 0 and toks.max() < vocab_size))):
        raise ValueError("an entry of the step is out of range")       # (plan_step says which)

    def runs_of(size):
        """-> (first rows, counts, first run of each portion) of the portions cut into runs of up to `size` tokens"""
        if base == len(lens):
            return row0, counts, row0
        runs = -(-counts // size)
        first = np.cumsum(runs) - runs
        off = size * (np.arange(int(runs.sum())) - np.repeat(first, runs))      # of a run inside its portion
        return ((np.repeat(row0, runs) + off).astype(i32), np.minimum(size, np.repeat(counts, runs) - off).astype(i32), first.astype(i32))
    tile_row0, tile_cnt, seq_tile0 = runs_of(StepPlan.TILE)
    chunk_row0, chunk_cnt, seq_chunk0 = runs_of(StepPlan.CHUNK)
    tok_start = np.repeat(starts, counts)
    return StepPlan(tile_row0=tile_row0, tile_cnt=tile_cnt, seq_cnt=counts, chunk_row0=chunk_row0, chunk_cnt=chunk_cnt,
                    seq_chunk0=seq_chunk0, seq_tile0=seq_tile0, seq_row0=row0, tok_start=tok_start,
                    tok_state=np.zeros(base, dtype=i32),
                    num_tokens=base, num_seqs=len(seq_ids), seq_ids_list=seq_ids, target_lens_list=targets,
                    input_ids=toks.astype(i32), tok_pos=(np.repeat(starts - row0, counts) + np.arange(base)).astype(i32),
                    tok_seq=np.repeat(np.asarray(seq_ids, dtype=i32), counts), want_rows=np.asarray(want, dtype=i32))
