"""Split decode steps on both sides of the rule by which every workgroup of a KV
group scores the group's pages itself (up to 160 pages) or a scoring launch does it
for all: page counts at the line, INT4 and INT8, every head ratio, both selection
modes, and the query layouts the in-kernel scorer reads in different ways (16-byte
aligned 16-bit rows, float32, rows off a 16-byte address, a transposed buffer).
Selection bit for bit against the oracle, O within the decode bar, lse within 1e-4."""
import numpy as np
import pytest
import torch

from oracle import fq_oracle as O
from tests.cases import Int4Case, Int8Case, decode_tol, max_err

pytestmark = pytest.mark.gpu


def _layout(q, how):
    B, H, _, D = q.shape
    if how == "offset":        # rows 2 bytes past a 16-byte address
        buf = torch.empty(B, H, 1, D + 8, dtype=q.dtype, device=q.device)
        buf[..., 1:D + 1] = q
        return buf[..., 1:D + 1]
    if how == "transposed":    # channel stride H
        return q.transpose(1, 3).contiguous().transpose(1, 3)
    return q


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("P,nrep,Hkv,B,mode,dtype,meta,how", [
    (160, 3, 8, 1, "per_q_head", "bf16", "bf16", "plain"), (161, 3, 8, 1, "per_q_head", "bf16", "bf16", "plain"),
    (160, 4, 2, 2, "per_kv_head_sum", "f16", "f16", "offset"), (161, 4, 2, 2, "per_kv_head_sum", "f16", "f16", "offset"),
    (129, 2, 3, 1, "per_q_head", "bf16", "bf16", "transposed"), (128, 1, 4, 1, "per_q_head", "f32", "bf16", "plain"),
    (97, 6, 2, 1, "per_q_head", "bf16", "bf16", "plain"), (160, 6, 2, 1, "per_kv_head_sum", "bf16", "bf16", "offset"),
    (161, 8, 2, 1, "per_kv_head_sum", "bf16", "bf16", "plain"), (160, 8, 2, 1, "per_q_head", "f32", "f16", "transposed"),
    (65, 3, 16, 8, "per_q_head", "bf16", "bf16", "plain")])
def test_step(bits, P, nrep, Hkv, B, mode, dtype, meta, how):
    print(f"[split scoring] bits={bits} P={P} nrep={nrep} Hkv={Hkv} B={B} {mode} {dtype}/{meta} {how}", flush=True)
    from flashquest_amd.eager.decode import quest_decode_int4, quest_decode_int8
    S = 64 * (P - 1) + 1 + 7 * nrep
    kw = dict(seed=P + nrep, B=B, Hq=nrep * Hkv, Hkv=Hkv, S=S, dtype="bf16" if dtype == "f32" else dtype, meta=meta)
    sel = dict(retention=0.45, num_sinks=4, window_pages=2)
    if bits == 4:
        c, op = Int4Case(**kw), quest_decode_int4
        names, host = ("K_packed", "K_scale", "K_mn", "V_packed", "V_scale", "V_mn"), (c.kp, c.ks, c.km, c.vp, c.vs, c.vm)
    else:
        c, op = Int8Case(**kw), quest_decode_int8
        names, host = ("K_uint8", "K_scale", "K_mn", "V_uint8", "V_scale", "V_mn"), (c.ku, c.ks, c.km, c.vu, c.vs, c.vm)
    d = c.device()
    q = c.q_dev()
    q = _layout(q.float() if dtype == "f32" else q, how)
    ref = O.decode_step(c.Q, *host, mode=mode, bits=bits, **sel)
    for rep in range(2):       # without and with the mask written by the attention launch
        out = op(q, *[d[k] for k in names], select_mode=mode, return_selection=rep == 1, **sel)
        if rep:
            assert np.array_equal(out[2].cpu().numpy(), ref["mask"])
        assert max_err(out[0][:, :, 0], ref["O"]) <= decode_tol(ref["O"], "bf16")
        assert max_err(out[1][:, :, 0], ref["lse"]) <= 1e-4
