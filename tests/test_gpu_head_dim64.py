"""64-channel heads on the matrix-core decode kernels, against the oracle: every
head ratio (6 and 8 as virtual KV heads), V metadata per token and per 32
channels, both selection modes, few groups (split) and many (one workgroup per
group), a page count past the in-kernel selection, a partial last page, the
partial-page tail inside the kernel and (float32) beside it, and strided cache
views.  Selection bit for bit; O within the decode bar, lse within 1e-4."""
import numpy as np
import pytest
import torch

from oracle import fq_oracle as O
from tests.cases import Int4Case, Int8Case, decode_tol, max_err, to_dev_half

pytestmark = pytest.mark.gpu

SEL = dict(retention=0.25, num_sinks=4, window_pages=2)


def _make(bits, **kw):
    if bits == 8:
        kw.pop("vgroup", None)
        c = Int8Case(D=64, **kw)
        return c, [c.device()[k] for k in ("K_uint8", "K_scale", "K_mn", "V_uint8", "V_scale", "V_mn")], \
            (c.ku, c.ks, c.km, c.vu, c.vs, c.vm)
    c = Int4Case(D=64, **kw)
    return c, [c.device()[k] for k in ("K_packed", "K_scale", "K_mn", "V_packed", "V_scale", "V_mn")], \
        (c.kp, c.ks, c.km, c.vp, c.vs, c.vm)


def _decode(bits):
    from flashquest_amd.eager.decode import quest_decode_int4, quest_decode_int8
    return quest_decode_int4 if bits == 4 else quest_decode_int8


@pytest.mark.parametrize("bits,dtype,vgroup", [(4, "bf16", None), (4, "f16", 32), (4, "bf16", 32), (8, "bf16", None),
                                               (8, "f16", None)])
@pytest.mark.parametrize("nrep,Hkv,B,S,mode", [
    (1, 2, 1, 64 * 9 + 1, "per_q_head"), (2, 3, 2, 64 * 64, "per_kv_head_sum"), (3, 2, 1, 64 * 100 + 63, "per_q_head"),
    (4, 8, 1, 64 * 256 + 5, "per_q_head"), (4, 8, 24, 64 * 50, "per_kv_head_sum"), (4, 2, 1, 64 * 600 + 9, "per_q_head"),
    (6, 2, 1, 64 * 130, "per_kv_head_sum"), (8, 4, 2, 64 * 70 + 17, "per_q_head"), (3, 1, 1, 40, "per_q_head")])
def test_step(bits, dtype, vgroup, nrep, Hkv, B, S, mode):
    print(f"[head_dim 64] bits={bits} {dtype} vgroup={vgroup} nrep={nrep} Hkv={Hkv} B={B} S={S} {mode}", flush=True)
    c, planes, host = _make(bits, seed=S + nrep, B=B, Hq=nrep * Hkv, Hkv=Hkv, S=S, dtype=dtype, meta=dtype, vgroup=vgroup)
    o, lse, mask = _decode(bits)(c.q_dev(), *planes, select_mode=mode, return_selection=True, **SEL)
    torch.cuda.synchronize()
    ref = O.decode_step(c.Q, *host, mode=mode, bits=bits, **SEL)
    assert np.array_equal(mask.cpu().numpy(), ref["mask"])
    assert max_err(o[:, :, 0], ref["O"]) <= decode_tol(ref["O"], dtype)
    assert max_err(lse[:, :, 0], ref["lse"]) <= 1e-4


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("T,tdtype,P", [(1, "bf16", 256), (64, "bf16", 256), (37, "f16", 60), (37, "f32", 60), (9, "bf16", 600)])
def test_tail(bits, T, tdtype, P):
    c, planes, host = _make(bits, seed=T + P, B=2, Hq=8, Hkv=2, S=64 * P, dtype="bf16", meta="bf16")
    rng = np.random.default_rng(T)
    rnd = O.rounder(tdtype)
    kt, vt = (rnd(rng.standard_normal((2, 2, T, 64)).astype(np.float32)) for _ in range(2))
    dt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[tdtype]
    # rows of a 64-row staging buffer, as the caches keep them
    dev = []
    for t in (kt, vt):
        buf = torch.zeros(2, 2, 64, 64, dtype=dt, device="cuda:0")
        buf[:, :, :T] = torch.from_numpy(t).to("cuda:0", dt)
        dev.append(buf[:, :, :T])
    o, lse = _decode(bits)(c.q_dev(), *planes, K_tail=dev[0], V_tail=dev[1], **SEL)
    torch.cuda.synchronize()
    ref = O.decode_step(c.Q, *host, mode="per_q_head", bits=bits, **SEL)
    ot, lt = O.dense_attn_with_lse(c.Q, kt, vt)
    ro = O.merge_two_attentions(ref["O"], ref["lse"], ot, lt)
    m = np.maximum(ref["lse"], lt)
    # the three-operator form rounds the tail's output to bf16 once more
    extra = 0.0 if tdtype != "f32" and P <= 512 else 2.0 ** -8 * float(np.abs(ot).max())
    assert max_err(o[:, :, 0], ro) <= decode_tol(ro, "bf16") + extra
    assert max_err(lse[:, :, 0], m + np.log(np.exp(ref["lse"] - m) + np.exp(lt - m))) <= 1e-4


@pytest.mark.parametrize("bits", [4, 8])
def test_layers_strides_and_masks(bits):
    """A layer axis, views of buffers with room beyond the pages, and the mask operator over the same selection."""
    from flashquest_amd.kernel import flash_attn_sparse_fwd, flash_attn_sparse_int4_fwd
    S, L = 64 * 33, 2
    made = [_make(bits, seed=70 + l, B=2, Hq=8, Hkv=2, S=S, dtype="bf16", meta="bf16") for l in range(L)]
    views = []
    for i in range(6):
        t = torch.stack([m[1][i] for m in made])
        room = torch.zeros(*t.shape[:3], t.shape[3] + 64, t.shape[4], dtype=t.dtype, device=t.device)
        room[:, :, :, :t.shape[3]] = t
        views.append(room[:, :, :, :t.shape[3]])
    Q = torch.stack([m[0].q_dev() for m in made])
    o, lse, mask = _decode(bits)(Q, *views, return_selection=True, **SEL)
    op = flash_attn_sparse_int4_fwd if bits == 4 else flash_attn_sparse_fwd
    for l, (c, _, host) in enumerate(made):
        ref = O.decode_step(c.Q, *host, mode="per_q_head", bits=bits, **SEL)
        assert np.array_equal(mask[l].cpu().numpy(), ref["mask"])
        assert max_err(o[l, :, :, 0], ref["O"]) <= decode_tol(ref["O"], "bf16")
        om, lm = op(Q[l], *[views[i][l] for i in (0, 1, 2, 3, 4, 5)], selection_mask=mask[l].unsqueeze(2))
        assert max_err(om[:, :, 0], ref["O"]) <= decode_tol(ref["O"], "bf16")
        assert max_err(lm[:, :, 0], ref["lse"]) <= 1e-4


def _dequant64(host, bits, page=64):
    """The cache's keys and values in 64 bits."""
    kc, ks, km, vc, vs, vm = host
    if bits == 4:
        kc, vc = O.unpack_int4(kc), O.unpack_int4(vc)
    at = np.arange(kc.shape[2]) // page
    G = vs.shape[-1]
    wide = lambda x: np.repeat(x.astype(np.float64), vc.shape[-1] // G, axis=-1)
    return kc * ks.astype(np.float64)[:, :, at] + km.astype(np.float64)[:, :, at], vc * wide(vs) + wide(vm)


@pytest.mark.parametrize("bits,meta,vgroup", [(4, "f16", None), (4, "f16", 32), (4, "bf16", None), (4, "bf16", 32),
                                              (8, "bf16", None), (8, "f16", None)])
@pytest.mark.parametrize("form", ["plain", "v_1e-2", "v_1e-3", "v_four_decades", "v_one_large_row", "q_two_decades"])
def test_operands_as_close_as_fp32(bits, meta, vgroup, form):
    """float32 queries against 64 bits, the error relative to |O| of each head, every page selected.

    The logits (log2 domain) stay below 32, where half an fp32 ulp is 2^-20: the
    rounded query, the sum of the products, the one with the page minimum and the
    difference to the maximum are four such roundings, each at most 2^-20 ln 2 of
    its token's weight.  They differ from token to token; a head whose weight lies
    on a single token keeps none of it (the normaliser has the same factor).  The
    sums of p v and of p then add 8 roundings of 2^-24.  Operands of 22 bits,
    p * V_scale held against a fixed or distant bound, or products summed with
    16-bit alignment are 6e-6 to 9e-2 here.
    """
    bound = 4 * 2.0 ** -20 * np.log(2) + 8 * 2.0 ** -24
    rng = np.random.default_rng(len(form) + bits)
    B, Hkv, nrep, S, D = 1, 2, 4, 64 * 40 + 21, 64
    K = 2 * rng.standard_normal((B, Hkv, S, D)).astype(np.float32)
    V = rng.standard_normal((B, Hkv, S, D)).astype(np.float32)
    Q = rng.standard_normal((B, Hkv * nrep, D)).astype(np.float32)
    if form.startswith("v_1e"):
        V *= np.float32(form[2:])
    elif form == "v_four_decades":
        V *= (10.0 ** -rng.uniform(0, 4, (B, Hkv, S, 1))).astype(np.float32)
    elif form == "v_one_large_row":
        V[:, :, S // 3] *= 300
    elif form == "q_two_decades":
        Q *= (10.0 ** -rng.uniform(0, 2, (B, Hkv * nrep, 1))).astype(np.float32)
    dt = torch.float16 if meta == "f16" else torch.bfloat16
    up = lambda a: torch.from_numpy(a).to("cuda:0")
    if bits == 4:
        host = (*O.quantize_k_int4(K, 64, "f32", meta), *O.quantize_v_int4(V, vgroup, meta))
    else:
        host = (*O.quantize_k_int8(K, 64, "f32", meta), *O.quantize_v_int8(V, meta))
    planes = [up(a) if i in (0, 3) else to_dev_half(a, meta) for i, a in enumerate(host)]
    K64, V64 = (np.repeat(x, nrep, axis=1) for x in _dequant64(host, bits))
    z = np.einsum("bhd,bhsd->bhs", Q.astype(np.float64), K64) / 8.0
    assert np.abs(z).max() * np.log2(np.e) < 32
    p = np.exp(z - z.max(-1, keepdims=True))
    want = np.einsum("bhs,bhsd->bhd", p, V64) / p.sum(-1)[..., None]
    lse64 = z.max(-1) + np.log(p.sum(-1))

    def close(o, lse):
        got = o[:, :, 0].double().cpu().numpy()
        err = np.linalg.norm(got - want, axis=-1) / np.linalg.norm(want, axis=-1)
        assert err.max() <= bound, (form, err.max())
        # the logits' four roundings, and lse's own (below 32)
        assert np.abs(lse[:, :, 0].double().cpu().numpy() - lse64).max() <= 4 * 2.0 ** -20 * np.log(2) + 2.0 ** -20

    q = up(Q)[:, :, None]
    o, lse = _decode(bits)(q, *planes, retention=1.0)
    assert o.dtype == torch.float32
    close(o, lse)
    from flashquest_amd.kernel import flash_attn_sparse_fwd, flash_attn_sparse_int4_fwd
    every = torch.ones(B, Hkv * nrep, 1, planes[1].shape[2], dtype=torch.bool, device="cuda:0")
    op = flash_attn_sparse_fwd if bits == 8 else flash_attn_sparse_int4_fwd
    close(*op(q, *planes, selection_mask=every))
