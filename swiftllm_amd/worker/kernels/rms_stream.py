"""fp32 residual stream with RMS norms, gated sublayer results and causal input convolutions with carried state.
csrc/rms_stream.hip."""
import torch

from swiftllm_amd import _hip

from .linear import SplitKPartials


def gated_add_rmsnorm(x: torch.Tensor, m: torch.Tensor = None, post: torch.Tensor = None, gate: torch.Tensor = None,
                      gate_bias: torch.Tensor = None, m2: torch.Tensor = None, m2_gate: torch.Tensor = None,
                      pre: torch.Tensor = None, eps: float = 1e-6, out_dtype: torch.dtype = None,
                      row_idx: torch.Tensor = None, conv=None):
    """In place on the fp32 stream x [T, width]:
        y = m (+ sigmoid(m2_gate[t]) * m2);  y *= sigmoid(gate + gate_bias);  x += y / rms(y) * post
    and returns x / rms(x) * pre in out_dtype when `pre` is given (of rows row_idx only, when given; then m must be None).
    `gate` and `m2_gate` may be column slices of wider matrices (row stride taken from the tensor). m may be a product's SplitKPartials, whose
    fp32 slabs are summed here. With `conv` (ConvInput; only where conv.fits(x), without row_idx) -> (that, its
    causal_conv_state with add_input), the convolution in the same launch where the rows' addresses allow it."""
    _hip.require_gpu_tensor(x, "x")
    n, width = x.shape
    assert x.dtype == torch.float32 and x.is_contiguous()
    dtype = m.dtype if m is not None else out_dtype
    if isinstance(m, SplitKPartials):
        assert m.shape == (n, width)
        quads = _quads(x, m.slabs, m2, gate, gate_bias, post, pre)
        if width % 4 or width > 8192 or not quads or (gate is not None and gate.stride(0) % 4):
            m = m.materialize()
    parts = m if isinstance(m, SplitKPartials) else None
    if m is not None:
        assert parts is not None or (m.shape == x.shape and m.is_contiguous())
        assert post is not None and post.dtype == torch.float32
        assert gate is None or (gate.shape == x.shape and gate.stride(1) == 1 and gate.dtype == dtype
                                and gate_bias.dtype == torch.float32 and gate_bias.numel() == width)
        assert m2 is None or (m2.shape == x.shape and m2.is_contiguous() and m2.dtype == dtype
                              and m2_gate.shape[0] == n and m2_gate.dtype == dtype)
    rows = n if row_idx is None else row_idx.shape[0]
    out = torch.empty((rows, width), dtype=dtype, device=x.device) if pre is not None else None
    if m is None and pre is None:
        return None
    fused = conv is not None and (gate is None or gate.stride(0) % 4 == 0) and _quads(x, None if m is None else m.slabs if parts is not None else m,
                                                                                      m2, gate, gate_bias, post, pre)
    if conv is not None:
        assert row_idx is None and pre is not None and conv.fits(x)
    rest = (_hip.ptr(m2), _hip.ptr(m2_gate), m2_gate.stride(0) if m2_gate is not None else 0, _hip.ptr(gate),
            gate.stride(0) if gate is not None else 0, _hip.ptr(gate_bias), _hip.ptr(post), _hip.ptr(out), _hip.ptr(pre))
    tail = (float(eps), rows, width, _hip.dtype_code3(dtype), _hip.stream())
    if fused:
        st, total = conv.st, torch.empty_like(out)
        _hip.call("swl_gated_add_rmsnorm_conv", _hip.ptr(x), 0 if parts is not None else _hip.ptr(m), 0 if parts is None else _hip.ptr(parts.slabs),
                  0 if parts is None else parts.k_splits, *rest, _hip.ptr(total), _hip.ptr(conv.w), conv.w.shape[0], _hip.ptr(st.pool),
                  st.pool.stride(0), int(conv.tail_off), _hip.ptr(st.tok_pos), _hip.ptr(st.tok_state), *tail)
        return out, total
    if parts is not None:
        assert row_idx is None
        _hip.call("swl_gated_add_rmsnorm_parts", _hip.ptr(x), _hip.ptr(parts.slabs), parts.k_splits, *rest, *tail)
    else:
        _hip.call("swl_gated_add_rmsnorm", _hip.ptr(x), _hip.ptr(m), *rest, _hip.ptr(row_idx), *tail)
    return out if conv is None else (out, causal_conv_state(out, conv.w, conv.st, conv.tail_off, add_input=True))


def _quads(*tensors) -> bool:
    """Whether each starts on four of its elements (None: no such operand)."""
    return all(t is None or t.data_ptr() % (4 * t.element_size()) == 0 for t in tensors)


def post_norm_add(x: torch.Tensor, a: torch.Tensor, post: torch.Tensor, b: torch.Tensor = None, a_norm: torch.Tensor = None,
                  b_norm: torch.Tensor = None, coef: float = 1.0, pre: torch.Tensor = None, eps: float = 1e-6,
                  want_out: bool = True):
    """In place on the fp32 stream x [T, width], for models whose sublayers read the stream itself:
        y = coef * (a' + b');  x += y / rms(y) * post
    with a' = a / rms(a) * a_norm when a_norm is given (else a), b' likewise (b optional). Returns the next sublayer's input
    in a's dtype: x itself, or x / rms(x) * pre when `pre` is given (None when not wanted)."""
    _hip.require_gpu_tensor(x, "x")
    n, width = x.shape
    assert x.dtype == torch.float32 and x.is_contiguous() and a.shape == x.shape and a.is_contiguous()
    assert b is None or (b.shape == x.shape and b.is_contiguous() and b.dtype == a.dtype)
    for w in (post, a_norm, b_norm, pre):
        assert w is None or (w.dtype == torch.float32 and w.is_contiguous() and w.numel() == width)
    out = torch.empty((n, width), dtype=a.dtype, device=x.device) if want_out else None
    _hip.call("swl_post_norm_add", _hip.ptr(x), _hip.ptr(a), _hip.ptr(a_norm), _hip.ptr(b), _hip.ptr(b_norm), float(coef),
              _hip.ptr(post), _hip.ptr(out), _hip.ptr(pre) if want_out else 0, float(eps), n, width,
              _hip.dtype_code3(a.dtype), _hip.stream())
    return out


class StateRef:
    """Where a step's kernels find per-sequence state: the slot pool, and the plan's per-token arrays. tiles (tile_row0, tile_cnt,
    seq_tile0): the portions cut into runs of up to 16 tokens, for recurrences that run by tiles. longest: tokens of the longest
    portion, where the caller knows it."""
    __slots__ = ("pool", "tok_pos", "tok_start", "tok_state", "tok_seq", "seq_row0", "seq_cnt", "tiles", "longest")

    def __init__(self, pool, tok_pos, tok_start, tok_state, tok_seq, seq_row0, seq_cnt, tiles=None, longest=0):
        self.tiles, self.longest = tiles, longest
        self.pool, self.tok_pos, self.tok_start, self.tok_state = pool, tok_pos, tok_start, tok_state
        self.tok_seq, self.seq_row0, self.seq_cnt = tok_seq, seq_row0, seq_cnt


class ConvInput:
    """The input convolution of the next sublayer: what causal_conv_state takes beside the rows."""
    __slots__ = ("w", "st", "tail_off")
    MAX_TAPS, MAX_WIDTH = 4, 4096       # (swl_gated_add_rmsnorm_conv)

    def __init__(self, w: torch.Tensor, st: StateRef, tail_off: int):
        self.w, self.st, self.tail_off = w, st, tail_off

    def fits(self, x: torch.Tensor) -> bool:
        """Whether rows like x's may be convolved in the launch that norms them: every portion a single token, whose earlier inputs are
        all in the state slot."""
        w, st = self.w, self.st
        return (st.longest == 1 and w.dtype == torch.float32 and w.is_contiguous() and w.shape[0] <= self.MAX_TAPS and w.shape[1] == x.shape[1]
                and w.shape[1] <= self.MAX_WIDTH and w.shape[1] % 4 == 0 and st.pool.stride(0) % 4 == 0 and self.tail_off % 4 == 0
                and _quads(w, st.pool))


def token_shift_mix(h: torch.Tensor, mu: torch.Tensor, st: StateRef, tail_off: int) -> torch.Tensor:
    """-> [mixes, T, width]: h[t] + (h[t - 1] - h[t]) * mu[s] for every row of mu (fp32 [mixes, width]); zeros stand before a
    sequence's first token, and its last h is carried at `tail_off` inside the state slot."""
    _hip.require_gpu_tensor(h, "h")
    n, c = h.shape
    assert h.stride(1) == 1 and mu.dtype == torch.float32 and mu.is_contiguous() and mu.shape[1] == c
    out = torch.empty((mu.shape[0], n, c), dtype=h.dtype, device=h.device)
    _hip.call("swl_token_shift_mix", _hip.ptr(out), _hip.ptr(h), h.stride(0), _hip.ptr(mu), mu.shape[0], _hip.ptr(st.pool),
              st.pool.stride(0), int(tail_off), _hip.ptr(st.tok_pos), _hip.ptr(st.tok_start), _hip.ptr(st.tok_state),
              _hip.ptr(st.tok_seq), n, c, _hip.dtype_code3(h.dtype), _hip.stream())
    return out


def causal_conv_state(h: torch.Tensor, w: torch.Tensor, st: StateRef, tail_off: int, add_input: bool) -> torch.Tensor:
    """(h +) causal convolution of h over time per channel; w fp32, tap-major [taps, channels] (the last row multiplies the
    current token); the last taps - 1 inputs of every sequence are carried at `tail_off` inside its state slot."""
    _hip.require_gpu_tensor(h, "h")
    n, c = h.shape
    assert h.stride(1) == 1 and w.dtype == torch.float32 and w.is_contiguous() and w.shape[1] == c
    out = torch.empty((n, c), dtype=h.dtype, device=h.device)
    _hip.call("swl_causal_conv_state", _hip.ptr(out), out.stride(0), _hip.ptr(h), h.stride(0), _hip.ptr(w),
              _hip.ptr(st.pool), st.pool.stride(0), int(tail_off), _hip.ptr(st.tok_pos), _hip.ptr(st.tok_start),
              _hip.ptr(st.tok_state), _hip.ptr(st.tok_seq), n, c, w.shape[0], 1 if add_input else 0,
              _hip.dtype_code3(h.dtype), _hip.stream())
    return out
