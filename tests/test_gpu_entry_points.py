"""Entry points of the C interface that the workers reach through their more general forms: the same bits as those with one share, one
segment or the plain mask."""
import pytest
import torch

from swiftllm_amd import _hip

pytestmark = pytest.mark.gpu
H, G, D, DV, T, KEYS = 4, 2, 64, 64, 20, 75


def _attention(dtype):
    """T tokens at the end of one sequence of KEYS keys, as tiles of 16 and less."""
    g = torch.Generator(device="cuda").manual_seed(1)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")       # noqa: E731
    i32 = lambda xs: torch.tensor(xs, dtype=torch.int32, device="cuda")     # noqa: E731
    blocks = -(-KEYS // 16)
    pool = rand(blocks, 16 * G * (D + DV)).to(dtype)
    a = dict(out=torch.full((T, H * DV), 7.0, dtype=dtype, device="cuda"), q=rand(T, H * D).to(dtype), pool=pool,
             table=i32([list(range(blocks))]), seq=i32([0] * T), pos=i32(range(KEYS - T, KEYS)), talk=rand(H, H) / H, rel=rand(H, 30),
             r1=torch.rand(H, device="cuda"), r2=torch.rand(H, device="cuda"), pb=rand(H), row0=i32([0, 16]), cnt=i32([16, T - 16]),
             code=_hip.dtype_code3(dtype), blocks=blocks)
    a["kv"] = [pool.data_ptr(), pool.data_ptr() + 16 * G * D * pool.element_size()]
    return a


def _both(a, one, general):
    got = []
    for name, args in (one, general):
        a["out"].fill_(7.0)
        _hip.call(name, *[_hip.ptr(x) if x is None or isinstance(x, torch.Tensor) else x for x in args])
        got.append(a["out"].clone())
    assert torch.isfinite(got[0].float()).all() and not (got[0] == 7.0).all() and torch.equal(got[0], got[1])


@pytest.mark.parametrize("mixed", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_a_token_a_workgroup(dtype, mixed):
    a = _attention(dtype)
    talk, rel = (a["talk"], None) if mixed else (None, a["rel"])
    head = [a["out"], a["q"], *a["kv"], a["table"], a["seq"], a["pos"]]
    body = [talk, rel, 30 if rel is not None else 0, T, H, G, D, DV, H * D, 40, 0.125, 20.0, a["blocks"], a["pool"].stride(0)]
    plain = [0, None, G, 0, None, DV, H * DV, None, 0]      # (window, no sink, slopes or gate)
    stream = _hip.stream()
    general = ("swl_masked_attn_shares", head + body + plain + [1, None, a["code"], stream])
    _both(a, ("swl_masked_attn", head + body + plain + [a["code"], stream]), general)
    _both(a, ("swl_window_attn", head + body + [a["code"], stream]), general)
    vectors = [talk, a["r1"], a["r2"], a["pb"]]
    body = [T, H, G, D, DV, H * D, 40, 0.125, a["blocks"], a["pool"].stride(0)]
    _both(a, ("swl_sigmoid_attn", head + vectors + body + [a["code"], stream]),
          ("swl_sigmoid_attn_shares", head + vectors + body + [1, None, a["code"], stream]))


@pytest.mark.parametrize("mixed", [True, False])
@pytest.mark.parametrize("shares", [1, 3])
def test_attention_by_tiles(shares, mixed):
    a = _attention(torch.bfloat16)
    talk, rel = (a["talk"], None) if mixed else (None, a["rel"])
    scratch = torch.empty(shares * T * H * (DV + 2), device="cuda")
    args = [a["out"], a["q"], *a["kv"], a["table"], a["seq"], a["pos"], a["row0"], a["cnt"], talk, rel, 30 if rel is not None else 0, 2, H, G,
            D, DV, H * D, 40, 0.125, 20.0, a["blocks"], a["pool"].stride(0), shares, scratch, T]
    _both(a, ("swl_window_attn_tiles", args + [a["code"], _hip.stream()]),
          ("swl_masked_attn_tiles", args + [0, None, G, 0, 0, None, DV, H * DV, None, 0, a["code"], _hip.stream()]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_scan_in_one_segment(dtype):
    from test_gpu_lorulix import Slots
    d, dv, heads, n = 40, 24, 3, 50
    g = torch.Generator(device="cuda").manual_seed(2)
    rand = lambda *shape: torch.randn(*shape, generator=g, device="cuda")       # noqa: E731
    q, k, v = rand(n, heads * d).to(dtype), rand(n, heads * d).to(dtype), rand(n, heads * dv).to(dtype)
    decay, dskip = torch.rand(n, heads * d, generator=g, device="cuda"), rand(heads)
    tiles = [(0, 16), (16, 4), (20, 16), (36, 14)]
    row0, cnt = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in zip(*tiles))
    first = torch.tensor([0, 2], dtype=torch.int32, device="cuda")
    qd, kd = torch.empty(4, heads, 16, 48, device="cuda"), torch.empty(4, heads, 48, 16, device="cuda")
    total, intra = torch.empty(4, heads, 48, device="cuda"), torch.empty(4, heads, 256, device="cuda")
    p, stream, code = _hip.ptr, _hip.stream(), _hip.dtype_code3(dtype)
    _hip.call("swl_linear_chunks", p(qd), p(kd), p(total), p(intra), p(q), heads * d, p(k), heads * d, p(decay), heads * d, 1, 0, 0, 1.0,
              p(row0), p(cnt), 4, heads, heads, d, code, stream)
    results = []
    for name, more in (("swl_linear_scan", []), ("swl_linear_scan_segments", [1, 0, 0])):
        slots = Slots([heads * d * dv], num_slots=2)
        st = slots.ref([(0, 0, 20), (1, 0, 30)])
        o = torch.full((n, heads * dv), float("nan"), device="cuda")
        _hip.call(name, p(o), heads * dv, p(qd), p(kd), p(total), p(intra), p(v), heads * dv, p(dskip), p(st.pool), st.pool.stride(0),
                  slots.off[0], p(st.seq_row0), p(st.seq_cnt), p(first), p(st.tok_pos), p(st.tok_state), 2, heads, d, dv, *more, code, stream)
        results.append((o, st.pool[:, slots.off[0]:slots.off[0] + heads * d * dv].clone()))
    assert torch.isfinite(results[0][0]).all() and all(torch.equal(a, b) for a, b in zip(*results))
