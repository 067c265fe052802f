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
