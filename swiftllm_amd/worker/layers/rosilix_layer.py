"""The sublayers of a Rosilix layer, each a function from its normed input to its raw result; the post-norm into the fp32
stream and the next input norm are the model's fused step (kernels/rms_stream.py)."""
import torch

from ..kernels.latent import LatentAttention
from ..kernels.linear import ROWS_MAX_TOKENS, TILE_RELU2, linear_rows, linear_tile
from ..kernels.moe import relu_squared
from ..kernels.rope_kv import diff_head_combine, rope_and_store_kv
from ..kernels.window_attn import MASK_CHUNK, MASK_WINDOW, AttentionSpec, masked_attention
from .kekapel_layer import _project, _project_partials
from .lorulix_layer import StepContext


class RosilixDiffAttention:
    """(q | k | v | gate) projection -> rotary + KV store -> chunked attention of both score maps over the shared values
    (fp32 results) -> a1 - lambda a2, unit RMS per head, (1 - diff), head gate -> output projection."""

    def __init__(self, layer_config, weight, eps: float, skinny: bool, pool_slice, max_positions: int):
        mx = self.mixer = layer_config.mixer
        self.w, self.eps, self.skinny, self.pool_slice, self.max_positions = weight, eps, skinny, pool_slice, max_positions
        # the two maps as attention heads: map-major queries and keys, key head g over value head g mod G
        self.spec = AttentionSpec(2 * mx.num_q_heads, 2 * mx.num_kv_heads, mx.head_dim, mx.value_dim, mx.scale,
                                  window=mx.chunk, mask_kind=MASK_CHUNK, num_v_heads=mx.num_kv_heads, out_f32=True)

    def forward(self, h: torch.Tensor, ctx: StepContext) -> torch.Tensor:
        mx, w = self.mixer, self.w
        proj = _project(h, w.proj, self.skinny)
        rope_and_store_kv(proj, w.freq, mx.rot.dims, ctx.pool, self.pool_slice, ctx.block_table, ctx.tok_seq, ctx.tok_pos,
                          2 * mx.num_q_heads, 2 * mx.num_kv_heads, mx.num_kv_heads, mx.head_dim, mx.value_dim)
        if ctx.pool is None:    # memory profiling: the attention's output buffer without its reads
            maps = torch.zeros((h.shape[0], 2 * mx.o_size), dtype=torch.float32, device=h.device)
        else:
            maps = masked_attention(proj, ctx.pool, self.pool_slice, ctx.block_table, ctx.tok_seq, ctx.tok_pos, self.spec,
                                    ctx.tiles, self.max_positions, leave_shares=True)
        gate = proj[:, w.gate_col:w.gate_col + mx.num_q_heads]
        y = diff_head_combine(maps, gate, w.lam, 1.0 - mx.diff, self.eps, mx.num_q_heads, mx.value_dim, h.dtype)
        return _project_partials(y, w.o, self.skinny)


class RosilixLatentAttention:
    """(q | compressed kv | gate) projection -> rotary, latent norm and cache store -> attention over the cached rows with the heads'
    sinks, expanded or folded, and head gate (kernels/latent.py) -> output projection. A layer that reads another layer's cache
    projects queries and gates only."""

    def __init__(self, layer_config, weight, eps: float, skinny: bool, pool_slice, max_positions: int):
        mx = self.mixer = layer_config.mixer
        self.w, self.skinny = weight, skinny
        spec = AttentionSpec(mx.num_q_heads, 1, mx.kv_rank + mx.rot_dim, mx.kv_rank, mx.scale, window=0, mask_kind=MASK_WINDOW,
                             sink=weight.sink)
        self.attend = LatentAttention(mx, weight, spec, eps, pool_slice, max_positions, weight.dkv_col)

    def forward(self, h: torch.Tensor, ctx: StepContext) -> torch.Tensor:
        mx, w = self.mixer, self.w
        proj = _project(h, w.proj, self.skinny)
        y = self.attend(proj, proj[:, w.gate_col:w.gate_col + mx.num_q_heads], ctx)
        return _project_partials(y, w.o, self.skinny)


class RosilixFeedForward:
    """down(relu(up h)^2)."""

    def __init__(self, layer_config, weight, skinny: bool):
        self.mlp, self.w, self.skinny = layer_config.mlp, weight, skinny

    def forward(self, h: torch.Tensor, ctx: StepContext) -> torch.Tensor:
        y = linear_rows(h, self.w.up, relu2=True) if self.skinny and h.shape[0] <= ROWS_MAX_TOKENS else None
        if y is None and self.skinny:
            y = linear_tile(h, self.w.up, TILE_RELU2, self.mlp.ffn_inter_dim)
        if y is None:
            y = relu_squared(_project(h, self.w.up, self.skinny), self.mlp.ffn_inter_dim)
        return _project_partials(y, self.w.down, self.skinny)
