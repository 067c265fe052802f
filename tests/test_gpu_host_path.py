"""The native host path gives what the general (ctypes) path gives, bit for bit,
over the forms it takes, and leaves the others to it: layouts that need a copy,
queries that are not contiguous, tensor subclasses."""
import pytest
import torch

from flashquest_amd import _host
from tests.cases import Int4Case, Int8Case

pytestmark = pytest.mark.gpu


def _both(monkeypatch, call, native=True):
    """call() through the native path and without the module: the same results.  native: whether the module takes
    every call made of it (None: either); a call before warms the workspace, without which it takes none."""
    host = _host.module()
    assert host is not None, "the native host path is built with the library"
    call()
    answers = []
    with monkeypatch.context() as m:
        for name in ("decode", "prefill", "quantize"):
            m.setattr(host, name, lambda *a, f=getattr(host, name): answers.append(f(*a)) or answers[-1])
        got = call()
    assert answers and (native is None or all((x is not None) == native for x in answers))
    with monkeypatch.context() as m:
        m.setattr(_host, "_module", None)
        want = call()
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert (g is None) == (w is None)
        if g is not None:
            assert type(g) is type(w) and g.shape == w.shape and g.stride() == w.stride() and g.dtype == w.dtype
            assert torch.equal(g, w)


def _planes(bits, room=0, layers=0, D=128):
    case = (Int4Case if bits == 4 else Int8Case)(seed=5, B=2, Hq=6, Hkv=2, S=64 * 45, D=D)
    keys = ("K_packed", "K_scale", "K_mn", "V_packed", "V_scale", "V_mn") if bits == 4 else \
        ("K_uint8", "K_scale", "K_mn", "V_uint8", "V_scale", "V_mn")
    d, out = case.device(), []
    for k in keys:
        t = torch.nn.functional.pad(d[k], (0, 0, 0, room))[:, :, :d[k].shape[2]]
        out.append(torch.stack([t] * layers) if layers else t)
    q = case.q_dev()
    return (torch.stack([q] * layers) if layers else q), out


class Sub(torch.Tensor):
    pass


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("form", ["plain", "layers", "room", "tail", "no_lse", "q_strided", "q_subclass", "misaligned", "k_max",
                                  "d64", "d64_tail", "f32_query", "sum", "pattern", "layer_patterns", "head_retention"])
def test_decode(monkeypatch, bits, form):
    from flashquest_amd.eager.decode import quest_decode_int4, quest_decode_int8
    D = 64 if form.startswith("d64") else 128
    q, planes = _planes(bits, room=3 if form == "room" else 0, layers=2 if form in ("layers", "layer_patterns") else 0, D=D)
    kw = dict(retention=0.3)
    if form.endswith("tail"):
        kw.update(K_tail=torch.randn(2, 2, 64, D, device="cuda").bfloat16()[:, :, :11],
                  V_tail=torch.randn(2, 2, 64, D, device="cuda").bfloat16()[:, :, :11])
    elif form == "no_lse":
        kw["return_lse"] = False
    elif form == "q_strided":
        q = torch.stack([q, q], dim=-1)[..., 0]
    elif form == "q_subclass":
        q = q.as_subclass(Sub)
    elif form == "misaligned":
        flat = torch.empty(planes[0].numel() + 2, dtype=torch.uint8, device="cuda")
        planes[0] = flat[2:].view(planes[0].shape).copy_(planes[0])
    elif form == "k_max":
        kw["k_max_static"] = 7
    elif form == "f32_query":
        q = q.float() * 1.001
    elif form == "sum":
        kw["select_mode"] = "per_kv_head_sum"
    elif form == "pattern":
        kw["head_pattern"] = torch.tensor([True, False])
    elif form == "layer_patterns":
        kw["head_pattern"] = torch.tensor([[True, False], [False, True]])
    elif form == "head_retention":
        kw["retention"] = torch.linspace(0.1, 0.6, 6)
    op = quest_decode_int4 if bits == 4 else quest_decode_int8
    _both(monkeypatch, lambda: op(q, *planes, **kw), native=form not in ("q_strided", "q_subclass", "misaligned"))


@pytest.mark.parametrize("layers", [0, 2])
@pytest.mark.parametrize("mode", ["per_q_head", "per_kv_head_sum"])
def test_decode_turbo(monkeypatch, layers, mode):
    from flashquest_amd.eager.decode import quest_decode_turbo
    from tests.cases import to_dev_half
    from tests.test_gpu_turbo_forms import _case, _device
    S = 64 * 30 + 7
    Q, host, raw = _case(9, 2, 6, 2, S)
    planes = _device(host, S + 3) + [to_dev_half(r, "bf16") for r in raw]
    q = to_dev_half(Q, "bf16")[:, :, None]
    if layers:
        q, planes = torch.stack([q] * layers), [torch.stack([p] * layers) for p in planes]
    _both(monkeypatch, lambda: quest_decode_turbo(q, *planes, retention=0.3, select_mode=mode))


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("tail,dtype", [(0, torch.bfloat16), (9, torch.bfloat16), (9, torch.float16)])
def test_prefill(monkeypatch, bits, tail, dtype):
    from flashquest_amd.kernel import flash_attn_prefill_int4, flash_attn_prefill_int8
    _, planes = _planes(bits)
    q = torch.randn(2, 6, 50, 128, device="cuda").to(dtype)
    kt, vt = (torch.randn(2, 2, tail, 128, device="cuda").to(dtype) for _ in range(2))
    op = flash_attn_prefill_int4 if bits == 4 else flash_attn_prefill_int8
    _both(monkeypatch, lambda: (op(q, *planes, kt, vt, causal_offset=100),), native=dtype == torch.bfloat16)


@pytest.mark.parametrize("meta", [torch.bfloat16, torch.float16])
def test_quantisers(monkeypatch, meta):
    from flashquest_amd.kernel import quantize_k, quantize_k_int4, quantize_v, quantize_v_int4
    x = torch.randn(2, 3, 130, 128, device="cuda").bfloat16()
    for y in (x, x.transpose(0, 1), x[..., ::2]):
        _both(monkeypatch, lambda: quantize_k_int4(y, 64, meta_dtype=meta) + quantize_v_int4(y, meta_dtype=meta) +
              quantize_v_int4(y, v_group=32, meta_dtype=meta) + quantize_k(y, 64, meta_dtype=meta) +
              quantize_v(y, meta_dtype=meta))


def test_errors_are_the_general_paths():
    from flashquest_amd.eager.decode import quest_decode_int4
    from flashquest_amd.kernel import quantize_k_int4
    q, planes = _planes(4)
    with pytest.raises(ValueError):
        quest_decode_int4(q, *planes, retention=1.5)
    with pytest.raises(AssertionError):
        quest_decode_int4(q, *planes[:2], planes[2].half(), *planes[3:], retention=0.3)
    with pytest.raises(ValueError):
        quantize_k_int4(torch.zeros(1, 1, 64, 63, device="cuda").bfloat16(), 64)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("form,made", [("plain", 1), ("first_call", 1), ("q_strided", 1), ("q_subclass", 1), ("five_heads", 1),
                                       ("six_heads_chunked", 2), ("f32_tail_d64", 1)])
def test_retention_is_prepared_once(monkeypatch, bits, form, made):
    """A call that the native path leaves to the general one has its retention rows
    (copies and launches, with a head pattern) made once; chunked heads once a chunk."""
    from flashquest_amd import _lib, _ops
    from flashquest_amd.eager.decode import quest_decode_int4, quest_decode_int8
    heads = {"five_heads": 10, "six_heads_chunked": 12}.get(form, 6)
    D = 64 if form == "f32_tail_d64" else 128
    c = (Int4Case if bits == 4 else Int8Case)(seed=6, B=1, Hq=heads, Hkv=2, S=64 * (520 if form == "six_heads_chunked" else 45),
                                              D=D)
    q, planes = c.q_dev(), list(c.device().values())
    op = quest_decode_int4 if bits == 4 else quest_decode_int8
    kw = dict(retention=torch.full((heads,), 0.3), head_pattern=torch.tensor([True, False]))
    op(q, *planes, **kw)                     # the workspace is there
    if form == "first_call":
        monkeypatch.setattr(_lib, "_ws", {})
    elif form == "q_strided":
        q = torch.stack([q, q], dim=-1)[..., 0]
    elif form == "q_subclass":
        q = q.as_subclass(Sub)
    elif form == "f32_tail_d64":
        kw.update(K_tail=torch.randn(1, 2, 9, D, device="cuda"), V_tail=torch.randn(1, 2, 9, D, device="cuda"))
    calls, rows = [], _ops.retention_rows
    monkeypatch.setattr(_ops, "retention_rows", lambda *a: calls.append(a) or rows(*a))
    op(q, *planes, **kw)
    assert len(calls) == made


@pytest.mark.parametrize("bits", [4, 8, 3])
@pytest.mark.parametrize("nrep", [6, 8])
def test_whole_steps_of_6_and_8_heads_go_natively(monkeypatch, bits, nrep):
    """6 or 8 query heads per KV head that the library runs as one launch take the native path."""
    from flashquest_amd.eager.decode import quest_decode_int4, quest_decode_int8, quest_decode_turbo
    from tests.cases import to_dev_half
    from tests.test_gpu_turbo_forms import _case, _device
    B, Hkv = 13, 8                           # 104 KV heads: 208 virtual ones, past the 192 that fill the GPU
    if bits == 3:
        Q, host, raw = _case(5, B, nrep * Hkv, Hkv, 64 * 12)
        q = to_dev_half(Q, "bf16")[:, :, None]
        planes = _device(host, 64 * 12) + [to_dev_half(r, "bf16") for r in raw]
        op = quest_decode_turbo
    else:
        c = (Int4Case if bits == 4 else Int8Case)(seed=5, B=B, Hq=nrep * Hkv, Hkv=Hkv, S=64 * 12)
        q, planes = c.q_dev(), list(c.device().values())
        op = quest_decode_int4 if bits == 4 else quest_decode_int8
    op(q, *planes, retention=0.3)            # the workspace is there
    host, got = _host.module(), []
    decode = host.decode
    monkeypatch.setattr(host, "decode", lambda *a: got.append(decode(*a)) or got[-1])
    o, lse = op(q, *planes, retention=0.3)
    assert len(got) == 1 and got[0] is not None and got[0][0] is o
    monkeypatch.setattr(_host, "_module", None)
    want = op(q, *planes, retention=0.3)
    assert torch.equal(o, want[0]) and torch.equal(lse, want[1])


@pytest.mark.parametrize("k_max", [2 ** 31, 2 ** 32 + 1, 2 ** 63 - 1, 2 ** 70])
def test_a_bound_past_32_bits_bounds_nothing(monkeypatch, k_max):
    from flashquest_amd.eager.decode import quest_decode_int4
    q, planes = _planes(4)
    _both(monkeypatch, lambda: quest_decode_int4(q, *planes, retention=0.3, k_max_static=k_max))
    assert torch.equal(quest_decode_int4(q, *planes, retention=0.3, k_max_static=k_max)[0],
                       quest_decode_int4(q, *planes, retention=0.3)[0])
