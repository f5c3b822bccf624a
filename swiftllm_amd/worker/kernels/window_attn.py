"""Attention over the paged pool for models whose heads are coupled before the softmax: per-head q/k RMS norm fused with
the KV store, then sliding-window attention with tanh soft-capping and an [H, H] head-mixing matrix. Prompt portions (with
or without a cached prefix) and decoded tokens go through the same two launches: every token carries its block-table row
and its position. csrc/qknorm_kv.hip, csrc/window_attn.hip."""
import numpy as np
import torch

from swiftllm_amd import _hip


class PoolSlice:
    """Where one layer run keeps its keys and values inside the shared block pool: element offsets inside a block."""
    __slots__ = ("k_offset", "v_offset")

    def __init__(self, k_offset: int, v_offset: int):
        self.k_offset, self.v_offset = k_offset, v_offset


def qknorm_and_store_kv(qkv: torch.Tensor, q_norm: torch.Tensor, k_norm: torch.Tensor, pool: torch.Tensor,
                        pool_slice: PoolSlice, block_table: torch.Tensor, tok_seq: torch.Tensor, tok_pos: torch.Tensor,
                        mixer, eps: float):
    """qkv [T, q | k | v] of one fused projection: q heads normalised in place, k heads normalised into the pool, v heads
    copied into the pool. pool None (memory profiling): only the query norm."""
    _hip.require_gpu_tensor(qkv, "qkv")
    assert qkv.dim() == 2 and qkv.stride(1) == 1 and qkv.shape[1] == mixer.q_size + mixer.k_size + mixer.v_size
    assert q_norm.dtype == k_norm.dtype == torch.float32 and q_norm.numel() == k_norm.numel() == mixer.head_dim
    assert tok_pos.dtype == torch.int32 and tok_pos.shape[0] == qkv.shape[0]
    kp = vp = 0
    stride = 0
    if pool is not None:
        assert pool.is_contiguous() and pool.dtype == qkv.dtype and block_table.is_contiguous()
        assert tok_seq.dtype == torch.int32 and tok_seq.shape[0] == qkv.shape[0]
        esize = pool.element_size()
        kp = pool.data_ptr() + pool_slice.k_offset * esize
        vp = pool.data_ptr() + pool_slice.v_offset * esize
        stride = pool.shape[1]
    _hip.call("swl_qknorm_store_kv", _hip.ptr(qkv), _hip.ptr(q_norm), _hip.ptr(k_norm), kp, vp, _hip.ptr(block_table),
              _hip.ptr(tok_seq), _hip.ptr(tok_pos), qkv.shape[0], mixer.num_q_heads, mixer.num_kv_heads, mixer.head_dim,
              mixer.value_dim, qkv.stride(0), block_table.shape[1] if block_table is not None else 0, stride, float(eps),
              _hip.dtype_code3(qkv.dtype), _hip.stream())


def qknorm_full_and_store_kv(q_or_qkv: torch.Tensor, q_norm: torch.Tensor, k_norm: torch.Tensor, pool: torch.Tensor,
                             pool_slice: PoolSlice, block_table: torch.Tensor, tok_seq: torch.Tensor,
                             tok_pos: torch.Tensor, mixer, eps: float, store: bool):
    """Whole-projection RMS norms (a weight per element) with the position-dependent query multiplier of `mixer`
    (q_temp_coef, q_temp_every). store: the rows are [q | k | v] and k, v go to the pool; else the rows are queries only."""
    _hip.require_gpu_tensor(q_or_qkv, "qkv")
    width = mixer.q_size + ((mixer.k_size + mixer.v_size) if store else 0)
    assert q_or_qkv.dim() == 2 and q_or_qkv.stride(1) == 1 and q_or_qkv.shape[1] == width
    assert q_norm.dtype == torch.float32 and q_norm.numel() == mixer.q_size
    assert tok_pos.dtype == torch.int32 and tok_pos.shape[0] == q_or_qkv.shape[0]
    kp = vp = stride = 0
    if store and pool is not None:
        assert k_norm.dtype == torch.float32 and k_norm.numel() == mixer.k_size
        assert pool.is_contiguous() and pool.dtype == q_or_qkv.dtype and block_table.is_contiguous()
        esize = pool.element_size()
        kp = pool.data_ptr() + pool_slice.k_offset * esize
        vp = pool.data_ptr() + pool_slice.v_offset * esize
        stride = pool.shape[1]
    _hip.call("swl_qknorm_full_store_kv", _hip.ptr(q_or_qkv), _hip.ptr(q_norm), _hip.ptr(k_norm), kp, vp,
              _hip.ptr(block_table), _hip.ptr(tok_seq), _hip.ptr(tok_pos), q_or_qkv.shape[0], mixer.num_q_heads,
              mixer.num_kv_heads, mixer.head_dim, mixer.value_dim, q_or_qkv.stride(0),
              block_table.shape[1] if block_table is not None else 0, stride, float(eps), float(mixer.q_temp_coef),
              int(mixer.q_temp_every), _hip.dtype_code3(q_or_qkv.dtype), _hip.stream())


def qkv_bias_norm_store(qkv: torch.Tensor, q_b: torch.Tensor, k_b: torch.Tensor, v_b: torch.Tensor, q_norm: torch.Tensor,
                        k_norm: torch.Tensor, pool: torch.Tensor, pool_slice: PoolSlice, block_table: torch.Tensor,
                        tok_seq: torch.Tensor, tok_pos: torch.Tensor, mixer, eps: float, v_other: torch.Tensor = None,
                        mix: float = 0.0):
    """qkv [T, q | k | v] of one fused projection whose biases (fp32, optional) are still to be added: q heads biased and
    normed in place (q_norm / k_norm [dim] fp32 weights shared by the heads, None: unit RMS without a weight), k heads biased
    and normed into the pool, v biased, blended as (1 - mix) v + mix v_other[t] when v_other [T, kv_heads * vdim] (a column
    slice is fine) is given, and written both back into its columns and into the pool. pool None: no store."""
    _hip.require_gpu_tensor(qkv, "qkv")
    assert qkv.dim() == 2 and qkv.stride(1) == 1 and qkv.shape[1] >= mixer.q_size + mixer.k_size + mixer.v_size
    for t, size in ((q_b, mixer.q_size), (k_b, mixer.k_size), (v_b, mixer.v_size), (q_norm, mixer.head_dim),
                    (k_norm, mixer.head_dim)):
        assert t is None or (t.dtype == torch.float32 and t.is_contiguous() and t.numel() == size)
    assert tok_pos.dtype == torch.int32 and tok_pos.shape[0] == qkv.shape[0]
    assert v_other is None or (v_other.dtype == qkv.dtype and v_other.stride(1) == 1 and v_other.shape[0] == qkv.shape[0]
                               and v_other.shape[1] == mixer.v_size)
    kp = vp = stride = 0
    if pool is not None:
        assert pool.is_contiguous() and pool.dtype == qkv.dtype and block_table.is_contiguous()
        assert tok_seq.dtype == torch.int32 and tok_seq.shape[0] == qkv.shape[0]
        esize = pool.element_size()
        kp = pool.data_ptr() + pool_slice.k_offset * esize
        vp = pool.data_ptr() + pool_slice.v_offset * esize
        stride = pool.shape[1]
    _hip.call("swl_qkv_bias_norm_store", _hip.ptr(qkv), _hip.ptr(q_b), _hip.ptr(k_b), _hip.ptr(v_b), _hip.ptr(q_norm),
              _hip.ptr(k_norm), _hip.ptr(v_other), v_other.stride(0) if v_other is not None else 0, float(mix), kp, vp,
              _hip.ptr(block_table), _hip.ptr(tok_seq), _hip.ptr(tok_pos), qkv.shape[0], mixer.num_q_heads,
              mixer.num_kv_heads, mixer.head_dim, mixer.value_dim, qkv.stride(0),
              block_table.shape[1] if block_table is not None else 0, stride, float(eps), _hip.dtype_code3(qkv.dtype),
              _hip.stream())


class StepTiles(tuple):
    """(tile_row0, tile_cnt) of a step, and its spans: runs of up to 32 consecutive tokens of one portion (row0, cnt, and per token
    the position where its portion starts). longest: the longest sequence of the step (spans only: never under graph replay).
    span_order: the spans in the order to take them up (StepPlan.span_order; None: last to first). portions: (lengths after the step, tokens)
    of the sequences, on the host."""

    def __new__(cls, tile_row0, tile_cnt, spans=None, longest=0, span_order=None, portions=None):
        self = super().__new__(cls, (tile_row0, tile_cnt))
        self.spans, self.longest, self.span_order = spans, longest, span_order
        self._portions, self._keys = portions, None
        return self

    @classmethod
    def of(cls, dev):
        return cls(dev["tile_row0"], dev["tile_cnt"], (dev["chunk_row0"], dev["chunk_cnt"], dev["tok_start"]), dev.get("longest", 0),
                   dev.get("span_order"), dev.get("portions"))

    def keys(self, tokens: int):
        """(keys that the step's tokens see, summed; lengths of the sequences that bring fewer than eight tokens, summed). Made when first asked
        for, where the device is already at work on the step."""
        if self._keys is None:
            if self._portions is None:
                self._keys = tokens * self.longest, 0
            else:
                lens, cnt = np.asarray(self._portions[0], dtype=np.int64), np.asarray(self._portions[1], dtype=np.int64)
                self._keys = int((cnt * (2 * lens - cnt + 1)).sum()) // 2, int(lens[cnt < 8].sum())
        return self._keys


# A step whose spans hold this many tokens on average or more is a prompt step (a span of one token fills one of a workgroup's 128 rows a
# head). One-token steps stay with the tile kernel, whose launches may be captured. Measured here and by tiles of 16 queries, us a launch,
# bf16: 8 portions of 4 tokens at 500 keys, 8 heads of 128 over 2 with a bias 15 / 18, latent rows of 8 heads 29 / 27, 16 mixed heads
# 18 / 32; 64 portions of 4 at 2000 keys 51 / 118, 115 / 179, 53 / 157; 200 decoded tokens at 1000 keys beside one portion of 930 92 / 299,
# 359 / 755, 205 / 717; 30 at 3900 keys beside one of 200 56 / 157, 71 / 178, 44 / 123.
SPAN_MIN_TOKENS = 4


def span_shares(n: int, spans: int, H: int, G: int, dim: int, vdim: int, window: int, longest: int, row_keys: int, lone_keys: int) -> int:
    """Over how many workgroups the keys of every tile of a prompt step are shared out: 1, 2, 4, or 8 where all of them are on the chip at
    once. The longest walk of a workgroup and what a CU has to walk in all (us a page of 16 keys, the slower of the two is the launch's time)
    shrink and stay; shares cost a launch and, each, the partial results written and read. Measured at 196 steps of 200 to 8000 tokens,
    prompts alone and beside 1 to 30 decoded tokens at 0.8k to 8k keys, 4 to 40 heads of 64 to 576 columns over 1 to 8, windows of 256 to
    1024: 3 % above the best of 1, 2, 4 and 8 on average (by workgroups and the longest sequence alone: 12 %). us by
    shares, 8 heads of 128 over 2: 2000 tokens 40.7 (1), 43.6 (2), 43.4 (4), beside 30 at 3900 keys 74.0, 70.8, 62.7; 4 x 500 beside 8 at
    8000 keys 140, 115, 91; 8 x 200 11.0, 24.4, 29.3, beside one at 2000 keys 40.4, 36.0, 31.9."""
    narrow = dim + vdim <= 320      # (two workgroups of 64 rows a CU; wide rows: one of 128)
    rows, slots = (64, 2 * _NUM_CUS) if narrow else (128, _NUM_CUS)
    wide = (dim + 2 * vdim) / 1600
    walk_us, load_us = (0.2, 0.3) if narrow else (1.07 * wide, 1.9 * wide)
    queries = max(1, rows >> (H // G - 1).bit_length())     # of a workgroup
    if window > 0:
        longest, row_keys, lone_keys = min(longest, window), min(row_keys, n * window), min(lone_keys, spans * window)
    walk, load = walk_us * (longest // 16 + 1), load_us * (row_keys / queries + lone_keys) * G / 16 / slots
    share = n * H * (vdim + 2) * 8 / 6e6        # (6 TB/s)
    best, best_us = 1, max(walk, load)
    for splits in (2, 4, 8):
        us = max(walk / splits, load) + 9 + splits * share
        if us < best_us and (splits < 8 or 8 * G * max(n / queries, spans) <= slots):
            best, best_us = splits, us
    return best


def _span_launch(q, out, kp, vp, pool, block_table, tok_seq, tok_pos, tiles, H, G, GV, dim, vdim, window, mask_kind, scale, softcap,
                 rel=None, sink=None, slopes=None, out_f32=False, out_dim=None, gate=None) -> bool:
    """The prompt form (csrc/span_attn.hip) where it serves the step; False: nothing was launched."""
    spans = getattr(tiles, "spans", None)
    n = q.shape[0]
    if spans is None or n < SPAN_MIN_TOKENS * spans[0].shape[0] or q.dtype == torch.float32:
        return False
    if not _hip.load().swl_span_attn_supported(H, G, GV, dim, vdim, int(rel is not None), _hip.dtype_code(q.dtype)):
        return False
    if (q.data_ptr() | kp | vp) % 16 or q.stride(0) % 8 or pool.shape[1] % 8:      # 16-byte operand loads
        return False
    row0, cnt, start = spans
    splits = span_shares(n, row0.shape[0], H, G, dim, vdim, window, tiles.longest, *tiles.keys(n))
    splits, scratch = share_scratch(q.device, splits, n * H * (vdim + 2))
    _hip.call("swl_span_attn_ordered", _hip.ptr(tiles.span_order), tiles.longest, _hip.ptr(out), _hip.ptr(q), kp, vp,
              _hip.ptr(block_table), _hip.ptr(tok_seq), _hip.ptr(tok_pos), _hip.ptr(start), _hip.ptr(row0), _hip.ptr(cnt), _hip.ptr(rel), rel.shape[1] if rel is not None else 0, row0.shape[0],
              H, G, GV, dim, vdim, q.stride(0), window, mask_kind, float(scale), float(softcap), block_table.shape[1], pool.shape[1],
              splits, _hip.ptr(scratch), n, _hip.ptr(sink), int(out_f32), _hip.ptr(slopes), vdim if out_dim is None else out_dim,
              out.stride(0), _hip.ptr(gate), gate.stride(0) if gate is not None else 0, _hip.dtype_code(q.dtype), _hip.stream())
    return True


# Steps with at least this many tokens go to the matrix-core kernel (tiles of up to 16 queries; a decoded token is a tile of
# one: the matrix core is mostly padding there, but the kernel reads every page once with wide loads and shares a tile's pages
# out over several workgroups when there are few tiles).
TILES_MIN_TOKENS = 1
_NUM_CUS = 256


# A launch takes fewer shares rather than more scratch than this (which memory profiling sets aside: its step runs without a pool).
# The rules ask for 137 MiB at 512 value columns and 34 MiB at 128; only per-token steps of more than 64k value columns a token meet it.
SHARE_MAX_SCRATCH = 256 << 20


def share_scratch(device, splits: int, floats: int):
    """-> (key shares, their fp32 scratch of `floats` each; None for one share), of this call alone: the launch that fills it and the one that
    combines it run on the caller's stream, where the allocator hands the memory on afterwards; a captured graph keeps it in its own
    pool. (A buffer kept per device would be shared by the streams and threads that launch attention at the same time.)"""
    splits = max(1, min(splits, SHARE_MAX_SCRATCH // (4 * max(floats, 1))))
    return splits, torch.empty(splits * floats, dtype=torch.float32, device=device) if splits > 1 else None


def choose_key_splits(num_tiles: int, mixer, max_positions: int, slots: int = _NUM_CUS) -> int:
    """Workgroups per tile: enough to occupy the chip (`slots` workgroups) when a step has few tiles, never more than the
    pages a tile can see. A function of the tile count and the model only (not of positions), so a captured decode graph
    stays valid."""
    span = mixer.window if mixer.window > 0 else max_positions
    pages = span // 16 + 2
    return max(1, min(slots // max(num_tiles, 1), pages // 4, 16))


def token_key_splits(n: int, heads: int, vdim: int, mixer, max_positions: int, device):
    """Key shares of the per-token kernels (and their scratch): up to 16 while they leave at most four workgroups a CU — a chunk of 64
    keys is a chain of some microseconds, and a step of few tokens has nothing else to fill the chip with."""
    splits = choose_key_splits(n, mixer, max_positions, slots=4 * _NUM_CUS)
    return share_scratch(device, splits, n * heads * (vdim + 2))


def mix_launch(entry, q, out, kp, vp, pool, block_table, tok_seq, tok_pos, tiles, mixer, vectors, extra, floats) -> bool:
    """The prompt form of attention with mixed heads (csrc/mix_attn.hip) where it serves the step; False: nothing was launched.
    vectors: the fp32 arguments of `entry`, extra: its constants after the scale, floats: fp32 a share leaves per (token, head)."""
    spans = getattr(tiles, "spans", None)
    n, H = q.shape[0], mixer.num_q_heads
    if spans is None or n < SPAN_MIN_TOKENS * spans[0].shape[0] or q.dtype == torch.float32:
        return False
    if not _hip.load().swl_mix_attn_supported(H, mixer.num_kv_heads, mixer.head_dim, mixer.value_dim, _hip.dtype_code(q.dtype)):
        return False
    if (q.data_ptr() | kp | vp) % 16 or q.stride(0) % 8 or pool.shape[1] % 8:      # 16-byte operand loads
        return False
    row0, cnt = tiles
    # the registers allow one workgroup a CU: with fewer tiles than CUs, every tile's keys are shared out (at 2 and 4 workgroups a CU a
    # step of 1.4 thousand tokens at 16 heads of 128 gets no faster and 9 % slower: each has its own prologue and partial results)
    splits = choose_key_splits(row0.shape[0], mixer, tiles.longest)
    splits, scratch = share_scratch(q.device, splits, n * H * floats)
    _hip.call(entry, _hip.ptr(out), _hip.ptr(q), kp, vp, _hip.ptr(block_table), _hip.ptr(tok_seq), _hip.ptr(tok_pos),
              _hip.ptr(row0), _hip.ptr(cnt), *[_hip.ptr(t) for t in vectors], row0.shape[0], H, mixer.num_kv_heads, mixer.head_dim,
              mixer.value_dim, q.stride(0), mixer.window, float(mixer.scale), *extra, block_table.shape[1], pool.shape[1], splits,
              _hip.ptr(scratch), n, _hip.dtype_code(q.dtype), _hip.stream())
    return True


def tiles_supported(mixer, dtype: torch.dtype) -> bool:
    if dtype not in (torch.float16, torch.bfloat16):
        return False
    return bool(_hip.load().swl_window_attn_tiles_supported(mixer.num_q_heads, mixer.num_kv_heads, mixer.head_dim,
                                                            mixer.value_dim, _hip.dtype_code(dtype)))


def window_attention(qkv: torch.Tensor, talk: torch.Tensor, pool: torch.Tensor, pool_slice: PoolSlice,
                     block_table: torch.Tensor, tok_seq: torch.Tensor, tok_pos: torch.Tensor, mixer,
                     tiles=None, max_positions: int = 1 << 20, rel: torch.Tensor = None) -> torch.Tensor:
    """-> [T, heads * vdim]. The queries are the (already normalised) first columns of qkv; keys and values come from the
    pool, which already holds this step's tokens. `tiles` = (tile_row0, tile_cnt) device arrays: the step cut into runs of
    up to 16 consecutive tokens of one sequence — given, and the shape served, the matrix-core kernel runs. `talk` None: the
    heads are not mixed. `rel` (fp32 [heads, distances]): a bias added to head h's score at distance query - key."""
    _hip.require_gpu_tensor(qkv, "qkv")
    assert talk is None or (talk.dtype == torch.float32 and talk.is_contiguous()
                            and talk.shape == (mixer.num_q_heads, mixer.num_q_heads))
    assert rel is None or (rel.dtype == torch.float32 and rel.is_contiguous() and rel.shape[0] == mixer.num_q_heads)
    rel_len = rel.shape[1] if rel is not None else 0
    assert pool.is_contiguous() and pool.dtype == qkv.dtype
    n = qkv.shape[0]
    out = torch.empty((n, mixer.num_q_heads * mixer.value_dim), dtype=qkv.dtype, device=qkv.device)
    esize = pool.element_size()
    if talk is None and _span_launch(qkv, out, pool.data_ptr() + pool_slice.k_offset * esize,
                                     pool.data_ptr() + pool_slice.v_offset * esize, pool, block_table, tok_seq, tok_pos, tiles,
                                     mixer.num_q_heads, mixer.num_kv_heads, mixer.num_kv_heads, mixer.head_dim, mixer.value_dim,
                                     mixer.window, MASK_WINDOW, mixer.scale, mixer.softcap, rel=rel):
        return out
    if talk is not None and rel is None and mix_launch(
            "swl_mix_attn", qkv, out, pool.data_ptr() + pool_slice.k_offset * esize, pool.data_ptr() + pool_slice.v_offset * esize,
            pool, block_table, tok_seq, tok_pos, tiles, mixer, (talk,), (float(mixer.softcap),), mixer.value_dim + 2):
        return out
    if tiles is not None and n >= TILES_MIN_TOKENS and tiles_supported(mixer, qkv.dtype):
        row0, cnt = tiles
        heads = talk is None and head_rows(mixer, row0, n)
        splits = head_rows_splits(mixer, n, max_positions) if heads else choose_key_splits(row0.shape[0], mixer, max_positions)
        splits, scratch = share_scratch(qkv.device, splits, n * mixer.num_q_heads * (mixer.value_dim + 2))
        _hip.call("swl_masked_attn_tiles", _hip.ptr(out), _hip.ptr(qkv), pool.data_ptr() + pool_slice.k_offset * esize,
                  pool.data_ptr() + pool_slice.v_offset * esize, _hip.ptr(block_table), _hip.ptr(tok_seq),
                  _hip.ptr(tok_pos), _hip.ptr(row0), _hip.ptr(cnt), _hip.ptr(talk), _hip.ptr(rel), rel_len, row0.shape[0],
                  mixer.num_q_heads, mixer.num_kv_heads, mixer.head_dim, mixer.value_dim, qkv.stride(0), mixer.window,
                  float(mixer.scale), float(mixer.softcap), block_table.shape[1], pool.shape[1], splits, _hip.ptr(scratch), n,
                  MASK_WINDOW, 0, mixer.num_kv_heads, 0, -1 if heads else 0, 0, mixer.value_dim, out.stride(0), 0, 0,
                  _hip.dtype_code(qkv.dtype), _hip.stream())
        return out
    splits, scratch = token_key_splits(n, mixer.num_q_heads, mixer.value_dim, mixer, max_positions, qkv.device)
    _hip.call("swl_masked_attn_shares", _hip.ptr(out), _hip.ptr(qkv), pool.data_ptr() + pool_slice.k_offset * esize,
              pool.data_ptr() + pool_slice.v_offset * esize, _hip.ptr(block_table), _hip.ptr(tok_seq), _hip.ptr(tok_pos),
              _hip.ptr(talk), _hip.ptr(rel), rel_len, n, mixer.num_q_heads, mixer.num_kv_heads, mixer.head_dim,
              mixer.value_dim, qkv.stride(0), mixer.window, float(mixer.scale), float(mixer.softcap), block_table.shape[1],
              pool.shape[1], MASK_WINDOW, 0, mixer.num_kv_heads, 0, 0, mixer.value_dim, out.stride(0), 0, 0, splits,
              _hip.ptr(scratch), _hip.dtype_code3(qkv.dtype), _hip.stream())
    return out


# ---- the same loops with other masks and denominators -----------------------------------------------------------------------
MASK_WINDOW = 0     # keys [p - window + 1, p]
MASK_CHUNK = 1      # keys [floor(p / window) * window, p]


class AttentionSpec:
    """Shape and constants of one attention over the pool, as the kernels see it (which need not be how the design counts
    its heads: two score maps over shared values are 2 H query heads, 2 G key heads and G value heads).
    num_v_heads: value heads in a page; key head g reads value head g % num_v_heads. slopes: fp32 [num_q_heads], slope times the
    distance query - key is taken off the score, or None. out_dim: value columns that count (the pages' rows may be wider). window:
    sliding window or chunk size
    (mask_kind), 0 for every earlier key. sink: fp32 [num_q_heads] logits that join the denominators, or None."""
    __slots__ = ("num_q_heads", "num_kv_heads", "num_v_heads", "head_dim", "value_dim", "window", "mask_kind", "scale",
                 "softcap", "sink", "out_f32", "slopes", "out_dim")

    def __init__(self, num_q_heads, num_kv_heads, head_dim, value_dim, scale, window=0, mask_kind=MASK_WINDOW,
                 num_v_heads=None, softcap=0.0, sink=None, out_f32=False, slopes=None, out_dim=None):
        self.num_q_heads, self.num_kv_heads, self.head_dim, self.value_dim = num_q_heads, num_kv_heads, head_dim, value_dim
        self.num_v_heads = num_kv_heads if num_v_heads is None else num_v_heads
        self.window, self.mask_kind, self.scale, self.softcap, self.sink, self.out_f32 = \
            window, mask_kind, scale, softcap, sink, out_f32
        self.slopes, self.out_dim = slopes, value_dim if out_dim is None else out_dim


def masked_tiles_supported(spec: AttentionSpec, dtype: torch.dtype) -> bool:
    if dtype not in (torch.float16, torch.bfloat16):
        return False
    return bool(_hip.load().swl_masked_attn_tiles_supported(spec.num_q_heads, spec.num_kv_heads, spec.num_v_heads,
                                                            spec.head_dim, spec.value_dim, _hip.dtype_code(dtype)))


_row_sizes = {}     # (dim, vdim, dtype) -> served_row_sizes
PADDING_LIMIT = 2.5


def served_row_sizes(dim: int, vdim: int, dtype: torch.dtype):
    """Key and value row sizes (in elements) that a layer with heads of `dim` / `vdim` should use in the pool: the smallest ones at
    least as large that the matrix-core kernel is compiled for — rows are then padded with zeros, which change neither scores nor
    outputs — or (dim, vdim) itself where padding would cost more than PADDING_LIMIT times the arithmetic, or in fp32."""
    if dtype == torch.float32:
        return dim, vdim
    key = (dim, vdim, dtype)
    if key not in _row_sizes:
        best, lib, code = (dim, vdim), _hip.load(), _hip.dtype_code(dtype)
        cost = PADDING_LIMIT * (dim + vdim)
        for kd in range(-(-dim // 16) * 16, int(cost) + 1, 16):
            for vd in range(-(-vdim // 16) * 16, int(cost) - kd + 1, 16):
                if kd + vd < cost and lib.swl_masked_attn_tiles_supported(1, 1, 1, kd, vd, code):
                    best, cost = (kd, vd), kd + vd
        _row_sizes[key] = best
    return _row_sizes[key]


# From this many heads over a key head on, a step of single tokens runs with the heads on the matrix-core tile's rows
HEAD_ROWS_MIN_HEADS = 2
# One-wave workgroups: eight a CU. 32 requests at 1k keys, 4 layers: 636 us a step with tokens as rows (four-wave workgroups), 608, 575, 565,
# 580 us at 2, 4, 8, 16 a CU; 2 requests at 1.9k keys 546 against 495 to 504 us.
HEAD_ROWS_SLOTS = 8 * _NUM_CUS


def head_rows(spec, row0: torch.Tensor, n: int) -> bool:
    """Whether every tile is one token (a decode step) and enough heads read a key head: the tile's rows are then the heads."""
    return row0.shape[0] == n and spec.num_q_heads >= HEAD_ROWS_MIN_HEADS * spec.num_kv_heads


def head_rows_splits(spec, n: int, max_positions: int) -> int:
    groups = spec.num_kv_heads * -(-spec.num_q_heads // spec.num_kv_heads // 16)
    return choose_key_splits(n * groups, spec, max_positions, slots=HEAD_ROWS_SLOTS)


def choose_heads_per_group(spec: AttentionSpec) -> int:
    """Heads of one workgroup of the matrix-core kernel (four waves): as many per wave as keep a wave's query, key and value
    fragments and accumulators in registers, so that many or wide heads are shared out over several workgroups."""
    per_wave = max(1, 512 // (spec.head_dim + spec.value_dim))
    per_wave = 4 if per_wave >= 4 else 2 if per_wave >= 2 else 1
    return min(spec.num_q_heads, 4 * per_wave)


class KeyShares:
    """Results of attention whose keys were shared out over workgroups, not added up yet (csrc/attn_combine.h): fp32 [shares][tokens][heads]
    [columns], then a maximum and a sum for every one; natural: the maxima are not in base-2 units."""
    __slots__ = ("data", "shares", "natural")
    MOST, MAX_DIM = 32, 256     # (swl_diff_head_combine_shares)

    def __init__(self, data: torch.Tensor, shares: int, natural: bool):
        self.data, self.shares, self.natural = data, shares, natural

    @classmethod
    def serve(cls, splits: int, value_dim: int) -> bool:
        return 1 < splits <= cls.MOST and value_dim <= cls.MAX_DIM and value_dim % 4 == 0


def masked_attention(q: torch.Tensor, pool: torch.Tensor, pool_slice: PoolSlice, block_table: torch.Tensor,
                     tok_seq: torch.Tensor, tok_pos: torch.Tensor, spec: AttentionSpec, tiles=None,
                     max_positions: int = 1 << 20, out: torch.Tensor = None, gate: torch.Tensor = None, leave_shares: bool = False):
    """-> [T, num_q_heads * out_dim] (fp32 when spec.out_f32, else q's dtype), written to `out` when given (a column slice of wider
    rows is fine), times sigmoid(gate) element by element when `gate` (likewise) is. q: rows whose first num_q_heads * head_dim
    columns are the queries (a column slice of a wider matrix is fine); keys and values come from the pool, which already
    holds this step's tokens. leave_shares (without sink, gate and out): a caller that adds up key shares itself takes them as KeyShares
    where the keys are shared out."""
    _hip.require_gpu_tensor(q, "q")
    assert not leave_shares or (spec.sink is None and gate is None and out is None and spec.out_dim == spec.value_dim)
    assert q.dim() == 2 and q.stride(1) == 1 and q.shape[1] >= spec.num_q_heads * spec.head_dim
    assert pool.is_contiguous() and pool.dtype == q.dtype and tok_pos.dtype == torch.int32 and tok_seq.dtype == torch.int32
    sink = spec.sink
    assert sink is None or (sink.dtype == torch.float32 and sink.is_contiguous() and sink.numel() == spec.num_q_heads)
    n, cols = q.shape[0], spec.num_q_heads * spec.out_dim
    assert spec.slopes is None or (spec.slopes.dtype == torch.float32 and spec.slopes.numel() == spec.num_q_heads)
    if out is None:
        out = torch.empty((n, cols), dtype=torch.float32 if spec.out_f32 else q.dtype, device=q.device)
    assert out.shape == (n, cols) and out.stride(1) == 1 and (out.dtype == torch.float32 if spec.out_f32 else out.dtype == q.dtype)
    assert gate is None or (gate.shape == (n, cols) and gate.stride(1) == 1 and gate.dtype == q.dtype)
    gate_stride = gate.stride(0) if gate is not None else 0
    esize = pool.element_size()
    kp = pool.data_ptr() + pool_slice.k_offset * esize
    vp = pool.data_ptr() + pool_slice.v_offset * esize
    wide_ok = q.stride(0) % 4 == 0 and q.data_ptr() % 8 == 0 and kp % 8 == 0 and vp % 8 == 0 and pool.shape[1] % 4 == 0
    wide_ok = wide_ok and out.data_ptr() % (16 if spec.out_f32 else 8) == 0 and out.stride(0) % 4 == 0
    if wide_ok and _span_launch(q, out, kp, vp, pool, block_table, tok_seq, tok_pos, tiles, spec.num_q_heads, spec.num_kv_heads,
                                spec.num_v_heads, spec.head_dim, spec.value_dim, spec.window, spec.mask_kind, spec.scale,
                                spec.softcap, sink=sink, slopes=spec.slopes, out_f32=spec.out_f32, out_dim=spec.out_dim, gate=gate):
        return out
    if tiles is not None and wide_ok and masked_tiles_supported(spec, q.dtype):
        row0, cnt = tiles
        if head_rows(spec, row0, n):
            hpg, splits = -1, head_rows_splits(spec, n, max_positions)
        else:
            hpg = choose_heads_per_group(spec)
            groups = -(-spec.num_q_heads // hpg)
            splits = choose_key_splits(row0.shape[0] * groups, spec, max_positions)
        splits, scratch = share_scratch(q.device, splits, n * spec.num_q_heads * (spec.value_dim + 2))
        leave = leave_shares and KeyShares.serve(splits, spec.value_dim)
        _hip.call("swl_masked_attn_tiles", _hip.ptr(out), _hip.ptr(q), kp, vp, _hip.ptr(block_table), _hip.ptr(tok_seq),
                  _hip.ptr(tok_pos), _hip.ptr(row0), _hip.ptr(cnt), 0, 0, 0, row0.shape[0], spec.num_q_heads,
                  spec.num_kv_heads, spec.head_dim, spec.value_dim, q.stride(0), spec.window, float(spec.scale),
                  float(spec.softcap), block_table.shape[1], pool.shape[1], splits, _hip.ptr(scratch), n, spec.mask_kind,
                  _hip.ptr(sink), spec.num_v_heads, 2 if leave else 1 if spec.out_f32 else 0, hpg, _hip.ptr(spec.slopes), spec.out_dim,
                  out.stride(0), _hip.ptr(gate), gate_stride, _hip.dtype_code(q.dtype), _hip.stream())
        return KeyShares(scratch, splits, False) if leave else out
    splits, scratch = token_key_splits(n, spec.num_q_heads, spec.value_dim, spec, max_positions, q.device)
    leave = leave_shares and KeyShares.serve(splits, spec.value_dim)
    _hip.call("swl_masked_attn_shares", _hip.ptr(out), _hip.ptr(q), kp, vp, _hip.ptr(block_table), _hip.ptr(tok_seq),
              _hip.ptr(tok_pos), 0, 0, 0, n, spec.num_q_heads, spec.num_kv_heads, spec.head_dim, spec.value_dim, q.stride(0),
              spec.window, float(spec.scale), float(spec.softcap), block_table.shape[1], pool.shape[1], spec.mask_kind,
              _hip.ptr(sink), spec.num_v_heads, 2 if leave else 1 if spec.out_f32 else 0, _hip.ptr(spec.slopes), spec.out_dim, out.stride(0),
              _hip.ptr(gate), gate_stride, splits, _hip.ptr(scratch), _hip.dtype_code3(q.dtype), _hip.stream())
    return KeyShares(scratch, splits, True) if leave else out
