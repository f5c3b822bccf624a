"""The gated delta rule as a recurrent mixer with per-sequence state slots. csrc/delta_rule.hip."""
import torch

from swiftllm_amd import _hip

from .rms_stream import StateRef


# A step whose longest portion holds this many tokens walks by tiles. Walked token by token a portion costs 10 us and 0.3 to 0.37 us a token;
# by tiles (heads of 128, 8 heads, the step's launches together): 1 portion of 24 / 64 / 1000 tokens 14 / 16 / 82 us against 17 / 30 / 331;
# 16 of 24 / 48 / 64: 26 / 34 / 37 against 26 / 39 / 50; 30 decoded tokens beside one of 32 / 64 / 200: 33 / 34 / 46 against 36 / 48 / 99.
TILES_MIN_PORTION = 48
# Decoded tokens and other short portions cost a nearly empty tile each (16 heads of 128: 1.2 us by tiles, 0.5 us by tokens), which the longest
# portion has to make up for: one more token for every so many workgroups (heads x 16 columns) of portions beyond a portion per
# TILES_FULL_TOKENS tokens. 16 heads of 128, 100 decoded tokens beside one portion of 48 / 80 / 150: 131 / 133 / 136 us by tiles, 109 / 133 /
# 189 by tokens; 200 beside one of 100 / 150 / 200: 245 / 249 / 254 against 220 / 257 / 291; 32 heads, 50 portions of 64 alone 292 against 430,
# beside 100 / 200 decoded tokens 551 / 798 against 561 / 708. Over 635 steps (4 to 32 heads of 64 and 128, up to 250 portions) a choice costs at
# most 2 % more than by tokens (66 % without this rule).
TILES_WORKGROUPS_A_TOKEN, TILES_FULL_TOKENS = 160, 24
# Steps that would need more scratch than this (1.6 KiB a token and head of 128) walk token by token.
TILES_MAX_SCRATCH = 1 << 30


def worth_tiles(longest: int, portions: int, tokens: int, heads: int, vdim: int) -> bool:
    """Whether a step of these portions is walked by tiles."""
    short = portions - tokens / TILES_FULL_TOKENS
    return longest >= max(TILES_MIN_PORTION, short * heads * vdim / 16 / TILES_WORKGROUPS_A_TOKEN)


def most_tiles_scratch(num_tokens: int, portions: int, mixer) -> int:
    """The most scratch (bytes) that the walk by tiles takes for a step of these sizes, however the tokens are shared out."""
    tiles = num_tokens // 16 + min(portions, num_tokens)        # (every portion may end in a part of one)
    need = _hip.load().swl_delta_rule_tiles_scratch_bytes(tiles, mixer.num_heads, mixer.head_dim, mixer.value_dim)
    return min(need, TILES_MAX_SCRATCH)


def delta_rule_mixer(proj: torch.Tensor, conv_w: torch.Tensor, a_log: torch.Tensor, dt_bias: torch.Tensor,
                     norm_w: torch.Tensor, st: StateRef, tail_off: int, state_off: int, mixer, eps: float) -> torch.Tensor:
    """proj [T, q | k | v | gate | b | a] (one fused projection) -> [T, heads * vdim] in proj's dtype: short convolutions
    (conv_w tap-major [taps, q | k | v channels]) +
    SiLU, unit q / k, the token-by-token recurrence on the fp32 state [heads, dim, vdim] at `state_off` inside each
    sequence's slot, then per head o / rms(o) * norm_w * silu(gate)."""
    _hip.require_gpu_tensor(proj, "proj")
    n = proj.shape[0]
    H, G, d, dv = mixer.num_heads, mixer.num_kv_heads, mixer.head_dim, mixer.value_dim
    assert proj.stride(1) == 1 and proj.shape[1] == mixer.proj_size
    assert conv_w.dtype == torch.float32 and conv_w.is_contiguous() and conv_w.shape == (mixer.conv_taps, mixer.conv_channels)
    assert a_log.dtype == dt_bias.dtype == norm_w.dtype == torch.float32 and a_log.numel() == dt_bias.numel() == H
    assert norm_w.numel() == dv
    dev, f32 = proj.device, torch.float32
    qn = torch.empty((n, G * d), dtype=f32, device=dev)
    kn = torch.empty((n, G * d), dtype=f32, device=dev)
    kq = torch.empty((n, G), dtype=f32, device=dev)
    vv = torch.empty((n, H * dv), dtype=f32, device=dev)
    beta = torch.empty((n, H), dtype=f32, device=dev)
    decay = torch.empty((n, H), dtype=f32, device=dev)
    code, stream = _hip.dtype_code3(proj.dtype), _hip.stream()
    _hip.call("swl_delta_prep", _hip.ptr(qn), _hip.ptr(kn), _hip.ptr(kq), _hip.ptr(vv), _hip.ptr(beta), _hip.ptr(decay), _hip.ptr(proj),
              proj.stride(0), _hip.ptr(conv_w), _hip.ptr(a_log), _hip.ptr(dt_bias), _hip.ptr(st.pool), st.pool.stride(0),
              int(tail_off), _hip.ptr(st.tok_pos), _hip.ptr(st.tok_start), _hip.ptr(st.tok_state), _hip.ptr(st.tok_seq), n,
              H, G, d, dv, mixer.conv_taps, code, stream)
    o = torch.empty((n, H * dv), dtype=f32, device=dev)
    delta_rule_scan(o, qn, kn, kq, vv, beta, decay, st, state_off, H, G, d, dv)
    out = torch.empty((n, H * dv), dtype=proj.dtype, device=dev)
    gate = proj[:, mixer.conv_channels:mixer.conv_channels + H * dv]
    gated_head_rmsnorm(out, o, gate, norm_w, H, dv, eps)
    return out


def delta_rule_scan(o, qn, kn, kq, vv, beta, decay, st: StateRef, state_off: int, H: int, G: int, d: int, dv: int):
    """o [T, H * dv] and the states from what the prep left (all fp32)."""
    num_seqs = st.seq_row0.shape[0]
    scratch_bytes = 0
    if st.tiles is not None and worth_tiles(st.longest, num_seqs, o.shape[0], H, dv) and _hip.load().swl_delta_rule_tiles_supported(H, G, d, dv):
        scratch_bytes = _hip.load().swl_delta_rule_tiles_scratch_bytes(st.tiles[0].shape[0], H, d, dv)
    if 0 < scratch_bytes <= TILES_MAX_SCRATCH:
        row0, cnt, seq_tile0 = st.tiles
        scratch = torch.empty(scratch_bytes // 4, dtype=torch.float32, device=o.device)
        _hip.call("swl_delta_rule_tiles", _hip.ptr(o), _hip.ptr(qn), _hip.ptr(kn), _hip.ptr(vv), _hip.ptr(beta), _hip.ptr(decay),
                  _hip.ptr(st.pool), st.pool.stride(0), int(state_off), _hip.ptr(st.seq_row0), _hip.ptr(st.seq_cnt),
                  _hip.ptr(seq_tile0), _hip.ptr(row0), _hip.ptr(cnt), _hip.ptr(st.tok_pos), _hip.ptr(st.tok_state), num_seqs,
                  row0.shape[0], H, G, d, dv, _hip.ptr(scratch), _hip.stream())
        return
    _hip.call("swl_delta_rule", _hip.ptr(o), _hip.ptr(qn), _hip.ptr(kn), _hip.ptr(kq), _hip.ptr(vv), _hip.ptr(beta), _hip.ptr(decay),
              _hip.ptr(st.pool), st.pool.stride(0), int(state_off), _hip.ptr(st.seq_row0), _hip.ptr(st.seq_cnt),
              _hip.ptr(st.tok_pos), _hip.ptr(st.tok_state), num_seqs, H, G, d, dv, _hip.stream())


def gated_head_rmsnorm(out: torch.Tensor, o: torch.Tensor, gate: torch.Tensor, norm_w: torch.Tensor, num_heads: int, vdim: int,
                       eps: float, mult: float = 1.0):
    """out[t, h] = mult * o / rms(o over the head) * norm_w * silu(gate): o fp32 [T, heads * vdim], gate and out rows of the compute
    dtype (column slices are fine), norm_w fp32 with one row of vdim for all heads or one per head."""
    _hip.require_gpu_tensor(o, "o")
    n = o.shape[0]
    assert o.dtype == norm_w.dtype == torch.float32 and o.is_contiguous() and o.shape[1] == num_heads * vdim
    assert norm_w.is_contiguous() and norm_w.numel() in (vdim, num_heads * vdim)
    for t in (gate, out):
        assert t.shape == (n, num_heads * vdim) and t.stride(1) == 1 and t.dtype == out.dtype
    _hip.call("swl_gated_head_rmsnorm", _hip.ptr(out), out.stride(0), _hip.ptr(o), _hip.ptr(gate), gate.stride(0),
              _hip.ptr(norm_w), vdim if norm_w.numel() != vdim else 0, float(mult), float(eps), n, num_heads, vdim,
              _hip.dtype_code3(out.dtype), _hip.stream())
