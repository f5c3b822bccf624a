"""Latent attention of a step: which rows run on the heads' own keys and values, expanded from the cached rows
(csrc/latent_expand.hip), and which on queries folded through the key up-projection — single tokens in three launches of their own
(csrc/latent_decode.hip)."""
import torch

from swiftllm_amd import _hip

from ..batch_plan import LatentExpansion
from .rope_kv import head_gate_, latent_rope_and_store_kv
from .window_attn import MASK_WINDOW, SHARE_MAX_SCRATCH, AttentionSpec, PoolSlice, StepTiles, choose_key_splits, masked_attention

# A layer's expanded pages take at most this much (which memory profiling sets aside: its step runs without a pool); portions past it stay
# folded. 8192 tokens of 16 heads of 128 + 64 and 128 columns take 80 MiB.
EXPAND_MAX_SCRATCH = 256 << 20
# (token, head) pairs that portions take beside others that stay folded. Two ways through attention are three launches more a layer, which the
# host, not the device, has to find time for in steps below about a millisecond. Two prompts beside 16 decoded tokens, us a pass, all folded
# and split: 2048 wide, 16 heads 2 x 16 924, 1057; 2 x 250 1038, 1098; 2 x 400 1060, 1120; 2 x 682 1242, 1173; 2 x 1000 1579, 1453; 1024 wide, 8 heads
# 2 x 250 1042, 1085; 2 x 1000 1093, 1131.
EXPAND_MIN_BESIDE = 18 * 1024


class ExpandedStep:
    """The device's side of a step's ExpandedPortions: `rows` leading rows on expanded pages, the rest folded."""
    __slots__ = ("rows", "pages", "page_row", "page_no", "page_dst", "tok_row", "table", "tiles", "rest")

    @classmethod
    def of(cls, dev):
        """From a step's views; None where every row stays folded."""
        ex = dev.get("expanded")
        if ex is None:
            return None
        self = cls()
        self.rows, self.pages = ex.rows, ex.pages
        self.page_row, self.page_no, self.page_dst = dev["ex_page_row"], dev["ex_page_no"], dev["ex_page_dst"]
        self.tok_row, self.table = dev["ex_tok_row"], dev["ex_table"].view(-1, 1)
        lens, cnt = dev["portions"]
        c0, t0, k = ex.chunks, ex.tiles, ex.seqs
        self.tiles = StepTiles(dev["tile_row0"][:t0], dev["tile_cnt"][:t0],
                               (dev["chunk_row0"][:c0], dev["chunk_cnt"][:c0], dev["tok_start"][:ex.rows]), int(max(lens[:k])),
                               dev["ex_order"] if "ex_order" in ex.arrays else None, (lens[:k], cnt[:k]))
        self.rest = None
        if k < len(lens):
            self.rest = StepTiles(dev["ex_rest_tile_row0"], dev["tile_cnt"][t0:],
                                  (dev["ex_rest_chunk_row0"], dev["chunk_cnt"][c0:], dev["tok_start"][ex.rows:]), int(max(lens[k:])),
                                  None, (lens[k:], cnt[k:]))
        return self


def latent_expansion(mixers, row_sizes, dtype: torch.dtype):
    """What decides for the steps of a model with these latent layers (LatentExpansion; None where no layer is served). row_sizes: of
    each layer's cached keys and values."""
    served = [mx for mx, (k_dim, _) in zip(mixers, row_sizes) if expansion_served(mx, k_dim, dtype)]
    if not served:
        return None
    page_bytes = max(2 * 16 * mx.num_q_heads * (mx.head_dim + mx.rot_dim + mx.value_dim) for mx in served)
    windows = [getattr(mx, "window", 0) for mx in served]
    mx = served[0]
    return LatentExpansion(mx.head_dim, mx.rot_dim, mx.value_dim, mx.kv_rank, 0 if 0 in windows else max(windows),
                           EXPAND_MAX_SCRATCH // page_bytes, EXPAND_MIN_BESIDE // mx.num_q_heads)


def expansion_served(mx, k_dim: int, dtype: torch.dtype) -> bool:
    if dtype not in (torch.float16, torch.bfloat16):
        return False
    lib, code, H = _hip.load(), _hip.dtype_code(dtype), mx.num_q_heads
    return bool(lib.swl_latent_expand_supported(mx.head_dim, mx.value_dim, mx.rot_dim, mx.kv_rank, k_dim, code)
                and lib.swl_span_attn_supported(H, H, H, mx.head_dim + mx.rot_dim, mx.value_dim, 0, code))


# Steps of up to this many tokens fold their queries beside the rotary and the store (one launch; the matrices are read once, a wave walks over
# the tokens); more go through a batched library product.
FOLD_MAX_TOKENS = 64


class LatentAttention:
    """The attention of a latent layer from its projected rows [query heads (dim | rot_dim) | ...] to the heads' gated results. spec: the
    folded attention (one key row of kv_rank + rot_dim and one value row of kv_rank for all heads).

    Single tokens, us of 32 at 1024 keys, 16 heads of 128 over rank 512 + 64, from the projection to the gated results: rotary and store 5.5, two
    batched products 4.2 and 9.2, attention of csrc/window_attn_mfma.hip 26, its combining launch 6.3, gate 4.7: 56; by csrc/latent_decode.hip
    6.6, 15.8 and 7.8: 30. That is made for rank 512 + 64 (swl_latent_decode_supported); other rows take the chain. All of it by tokens, heads
    and keys, chain / own launches: 1 x 16 x 1000 41 / 21; 64 x 8 x 300 46 / 28, x 4000 143 / 70; 64 x 40 x 1000 129 / 61; 256 x 16 x 300 93 / 57; 512 x
    16 x 40 79 / 76, x 1000 287 / 182; 256 x 40 x 40 91 / 94, x 300 165 / 128; 512 x 40 x 40 98 / 164, x 300 282 / 226: the value product reads a
    head's matrix for every four tokens, which only keys few enough not to matter let one see. (Counts alone decide, for captured steps, and cannot
    tell these apart.)"""

    def __init__(self, mixer, weight, spec: AttentionSpec, eps: float, pool_slice, max_positions: int, dkv_col: int):
        self.mixer, self.w, self.spec, self.eps, self.pool_slice, self.max_positions = mixer, weight, spec, eps, pool_slice, max_positions
        self.dkv_col = dkv_col
        H, dtype = mixer.num_q_heads, weight.uk.dtype
        self.heads_spec = AttentionSpec(H, H, mixer.head_dim + mixer.rot_dim, mixer.value_dim, spec.scale, window=spec.window,
                                        mask_kind=MASK_WINDOW, sink=spec.sink)
        self.expands = expansion_served(mixer, spec.head_dim, dtype)
        self.decodes = self.folds = False
        if dtype != torch.float32:
            lib, code = _hip.load(), _hip.dtype_code(dtype)
            self.decodes = bool(lib.swl_latent_decode_supported(mixer.kv_rank, mixer.rot_dim, spec.head_dim, mixer.value_dim, code))
            self.folds = self.decodes and bool(lib.swl_latent_fold_supported(mixer.head_dim, mixer.rot_dim, mixer.kv_rank, spec.head_dim, code))
        # the up-projections the other way round, where a kernel reads them; kept with the weights, which several runs of a layer share
        if self.folds and weight.uk_t is None:
            weight.uk_t = weight.uk.transpose(1, 2).contiguous()
        if (self.decodes or self.expands) and weight.uv is None:
            weight.uv = weight.uv_t.transpose(1, 2).contiguous()

    def __call__(self, proj: torch.Tensor, gate: torch.Tensor, ctx) -> torch.Tensor:
        """gate: [T, heads] logits, a column slice of the projected rows."""
        mx, w, sp = self.mixer, self.w, self.spec
        n, H, d, dr, r, e = proj.shape[0], mx.num_q_heads, mx.head_dim, mx.rot_dim, mx.kv_rank, mx.value_dim
        aligned = ctx.pool is not None and ctx.pool.shape[1] % 8 == 0 and self.pool_slice.k_offset % 8 == 0      # 16-byte loads of cached rows
        ex = ctx.expanded if self.expands and aligned else None
        m = ex.rows if ex is not None else 0
        tiles = ex.rest if m else ctx.tiles
        single = self.decodes and aligned and m < n and tiles is not None and tiles[0].shape[0] == n - m and \
            (n - m) * H * (r + 2) * 4 <= SHARE_MAX_SCRATCH
        qa = torch.empty((n - m, H * sp.head_dim), dtype=proj.dtype, device=proj.device)
        folded = single and m == 0 and self.folds and n <= FOLD_MAX_TOKENS and proj.data_ptr() % 16 == 0 and proj.stride(0) % 8 == 0
        if folded:
            self._fold(proj, qa, ctx)
        else:
            latent_rope_and_store_kv(proj, qa, w.freq, w.c_norm, ctx.pool, self.pool_slice, ctx.block_table, ctx.tok_seq,
                                     ctx.tok_pos, mx, self.dkv_col, self.eps, sp.head_dim, sp.value_dim, in_place=m)
        y = torch.empty((n, H * e), dtype=proj.dtype, device=proj.device)
        if m:
            self._expanded(proj, y[:m], ctx, ex)
        if m < n:
            # (views cost the host as much as a launch: none where every row is folded)
            part = (lambda t: t[m:]) if m else (lambda t: t)
            seq, pos, yr = part(ctx.tok_seq), part(ctx.tok_pos), part(y)
            if not folded:
                # q_abs[t, h, :] = W_uk,h^T q_unrotated[t, h, :]  -> the first kv_rank columns of every head of qa
                qn = part(proj)[:, :H * (d + dr)].view(n - m, H, d + dr)[:, :, :d].transpose(0, 1)       # [H, T, d]
                torch.bmm(qn, w.uk, out=qa.view(n - m, H, sp.head_dim)[:, :, :r].transpose(0, 1))   # (a strided batched product: no copy)
            if single:
                self._single(qa, yr, part(gate), ctx, seq, pos)
                if m:
                    head_gate_(y[:m], gate[:m], H, e)
                return y
            if ctx.pool is None:    # memory profiling: the attention's output buffer without its reads
                att = torch.zeros((n - m, H * sp.value_dim), dtype=proj.dtype, device=proj.device)
            else:
                att = masked_attention(qa, ctx.pool, self.pool_slice, ctx.block_table, seq, pos, sp, tiles, self.max_positions)
            torch.bmm(att.view(n - m, H, sp.value_dim)[:, :, :r].transpose(0, 1), w.uv_t, out=yr.view(n - m, H, e).transpose(0, 1))
        return head_gate_(y, gate, H, e)

    def _fold(self, proj, qa, ctx):
        mx, w, sp, esize = self.mixer, self.w, self.spec, proj.element_size()
        own = self.dkv_col >= 0
        kp, vp = (ctx.pool.data_ptr() + off * esize if own else 0 for off in (self.pool_slice.k_offset, self.pool_slice.v_offset))
        _hip.call("swl_latent_fold", _hip.ptr(proj), _hip.ptr(qa), _hip.ptr(w.uk_t), _hip.ptr(w.freq), _hip.ptr(w.c_norm), kp, vp,
                  _hip.ptr(ctx.block_table), _hip.ptr(ctx.tok_seq), _hip.ptr(ctx.tok_pos), proj.shape[0], mx.num_q_heads, mx.head_dim,
                  mx.rot_dim, mx.kv_rank, proj.stride(0), self.dkv_col if own else -1, qa.stride(0), ctx.block_table.shape[1],
                  ctx.pool.shape[1], float(self.eps), 1 if mx.rot.half else 0, float(mx.rot.multiplier), sp.head_dim, sp.value_dim,
                  _hip.dtype_code(proj.dtype), _hip.stream())

    def _single(self, qa, y, gate, ctx, seq, pos):
        mx, w, sp = self.mixer, self.w, self.spec
        n, H, code = qa.shape[0], mx.num_q_heads, _hip.dtype_code(qa.dtype)
        # (of the counts and the model alone: a captured step stays valid)
        floats = n * H * (mx.kv_rank + 2)
        shares = max(1, min(choose_key_splits(n * -(-H // 16), sp, self.max_positions), SHARE_MAX_SCRATCH // (4 * floats)))
        scratch = torch.empty(shares * floats, dtype=torch.float32, device=qa.device)
        _hip.call("swl_latent_decode", _hip.ptr(scratch), _hip.ptr(qa), ctx.pool.data_ptr() + self.pool_slice.k_offset * qa.element_size(),
                  _hip.ptr(ctx.block_table), _hip.ptr(seq), _hip.ptr(pos), n, H, qa.stride(0), sp.window,
                  float(sp.scale), ctx.block_table.shape[1], ctx.pool.shape[1], shares, code, _hip.stream())
        _hip.call("swl_latent_unfold", _hip.ptr(y), _hip.ptr(scratch), _hip.ptr(w.uv), _hip.ptr(sp.sink), _hip.ptr(gate), gate.stride(0), n, H,
                  mx.value_dim, shares, code, _hip.stream())

    def _expanded(self, proj, out, ctx, ex: ExpandedStep):
        mx, w, sp, hs = self.mixer, self.w, self.spec, self.heads_spec
        H, m, esize = mx.num_q_heads, ex.rows, proj.element_size()
        keys, values = 16 * H * hs.head_dim, 16 * H * mx.value_dim      # (elements of a page)
        pages = torch.empty((ex.pages, keys + values), dtype=proj.dtype, device=proj.device)
        _hip.call("swl_latent_expand", _hip.ptr(pages), ctx.pool.data_ptr() + self.pool_slice.k_offset * esize, _hip.ptr(w.uk),
                  _hip.ptr(w.uv), _hip.ptr(ctx.block_table), _hip.ptr(ex.page_row), _hip.ptr(ex.page_no), _hip.ptr(ex.page_dst),
                  ex.page_no.shape[0], H, mx.head_dim, mx.value_dim, mx.rot_dim, mx.kv_rank, sp.head_dim, ctx.block_table.shape[1],
                  ctx.pool.shape[1], _hip.dtype_code(proj.dtype), _hip.stream())
        masked_attention(proj[:m], pages, PoolSlice(0, keys), ex.table, ex.tok_row, ctx.tok_pos[:m], hs, ex.tiles, self.max_positions, out=out)
