"""The TurboQuant matrix-core decode over the forms it accepts: query types,
strided planes (rows of a longer buffer, also with an odd token count, so the
2-byte scales' rows start at any even address), page counts with a partial last
page, and V planes off a 4-byte address, which the general kernel takes.  Float32
results are held to the fixed point's own bound; a page whose scale is NaN and a
query that holds one must not pass for a number."""
import numpy as np
import pytest
import torch

from oracle import fq_oracle as O
from tests.cases import max_err, to_dev, to_dev_half

pytestmark = pytest.mark.gpu


def _case(seed, B, Hq, Hkv, S):
    rng = np.random.default_rng(seed)
    K, V = (rng.standard_normal((B, Hkv, S, 128)).astype(np.float32) for _ in range(2))
    V *= np.exp(rng.standard_normal((B, Hkv, S, 1))).astype(np.float32)         # V scales over some binades
    km, kl, ks, ksr, kmr = O.quantize_k_turbo(K, 64)
    vm, vl, vs = O.quantize_turbo(V)
    return rng.standard_normal((B, Hq, 128)).astype(np.float32), (km, kl, ks, vm, vl, vs), (ksr, kmr)


def _device(planes, rows, shift=0):
    """Planes as views of `rows`-token buffers whose bytes past S are junk."""
    out = []
    for i, a in enumerate(planes):
        t = to_dev(a) if i in (0, 1, 3, 4) else to_dev_half(a, "bf16")
        B, H, S, W = t.shape
        off = shift if i in (3, 4) else 0
        buf = torch.full((B * H * rows * W + 16,), 77, dtype=t.dtype, device="cuda")
        view = buf[off:off + B * H * rows * W].view(B, H, rows, W)
        view[:, :, :S] = t
        out.append(view[:, :, :S])
    return out


@pytest.mark.parametrize("rows,shift", [(0, 0), (1, 0), (5, 0), (64, 0), (0, 2)])
@pytest.mark.parametrize("dtype,Hq,Hkv,B,S", [("f32", 6, 2, 2, 64 * 9 + 1), ("f32", 4, 1, 1, 64 * 120 + 63), ("bf16", 3, 3, 1, 40),
                                              ("f16", 4, 2, 1, 64 * 30), ("f32", 6, 1, 1, 64 * 33 + 7)])
def test_forms(rows, shift, dtype, Hq, Hkv, B, S):
    from flashquest_amd.eager import quest_decode_turbo
    from flashquest_amd.kernel import flash_attn_sparse_turbo_fwd
    print(f"[turbo forms] rows=S+{rows} shift={shift} {dtype} Hq={Hq} Hkv={Hkv} B={B} S={S}", flush=True)
    Q, planes, raw = _case(S + Hq, B, Hq, Hkv, S)
    Q = O.rounder(dtype)(Q)
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    q = torch.from_numpy(Q).to("cuda", dt)[:, :, None]
    dev = _device(planes, S + rows, shift)
    meta = [to_dev_half(r, "bf16") for r in raw]
    o, lse, mask = quest_decode_turbo(q, *dev, *meta, retention=0.3, num_sinks=2, window_pages=1, select_mode="per_q_head",
                                      return_selection=True)
    o2, lse2 = flash_attn_sparse_turbo_fwd(q, *dev, selection_mask=mask[:, :, None])
    torch.cuda.synchronize()
    ref_mask = O.select_pages_vectorized(O.page_scores_fixed(Q, *raw, "per_q_head")[:, :, None, :],
                                         np.full(Hq, 0.3, np.float32), 2, 1)[:, :, 0, :]
    assert np.array_equal(mask.cpu().numpy(), ref_mask)
    ref_o, ref_l = O.sparse_turbo_attention(Q, *planes, ref_mask, 64)
    # a logit is off by the rotation's and the digits' rounding, at most 16 ulp of the largest |q_rot . k|
    # (|q_rot| < 5 and |k| < 5 here: 128 * 25 / sqrt(128) < 2^9), so a probability by 2^-11 of itself at worst
    # and 2^-17 in the mean; a p V product by 2^-24 of the largest V: O moves by less than 2^-15 of max |V|
    vmax = np.abs(O.dequant_turbo_rot(*planes[3:], 128)).max()
    bar = 2.0 ** -15 * vmax if dtype == "f32" else {"bf16": 2.0 ** -8, "f16": 2.0 ** -11}[dtype] * np.abs(ref_o).max() + 2.0 ** -15 * vmax
    for oo, ll in ((o, lse), (o2, lse2)):
        assert max_err(oo[:, :, 0], ref_o) <= bar
        assert max_err(ll[:, :, 0], ref_l) <= 1e-4


@pytest.mark.parametrize("where,value", [("q", float("nan")), ("q", float("inf")), ("k", float("nan")), ("v", float("nan")),
                                         ("v", float("inf"))])
def test_not_a_number(where, value):
    """As the float kernels treat them: a NaN or infinite query row and a NaN K scale leave no
    finite logit sum (lse -inf or NaN), V scales reach O; the other KV head is untouched."""
    from flashquest_amd.eager import quest_decode_turbo
    Q, planes, raw = _case(5, 1, 6, 2, 64 * 12)
    q = to_dev_half(Q, "bf16")[:, :, None]
    dev, meta = _device(planes, 64 * 12), [to_dev_half(r, "bf16") for r in raw]
    kw = dict(retention=1.0, num_sinks=1, window_pages=1)
    o, lse = quest_decode_turbo(q, *dev, *meta, **kw)
    {"q": q[0, 1], "k": dev[2][0, 0, 70], "v": dev[5][0, 0, 70]}[where].view(-1)[0] = value
    o2, lse2 = quest_decode_turbo(q, *dev, *meta, **kw)
    assert torch.equal(o[:, 3:], o2[:, 3:]) and torch.equal(lse[:, 3:], lse2[:, 3:])
    if where == "q":
        assert not lse2[0, 1].isfinite().any() and torch.equal(o[:, 0], o2[:, 0])
    elif where == "k":
        assert not lse2[0, :3].isfinite().any()
    else:
        assert not o2[0, :3].isfinite().any() and torch.equal(lse[:, :3], lse2[:, :3])
