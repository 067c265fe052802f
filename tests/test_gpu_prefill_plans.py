"""The dense prefill's forms (key groups per workgroup 1 / 2 / 4, with and
without key-range splits) against the CPU oracle: row counts around the 64-,
128- and 256-row blocks, key counts around the 128-key stages, whole prompts and
chunks over a cache, splits that leave the first row blocks' last slices empty.
Each shape names the form it takes (csrc/prefill.hip, dense_plan), which
test_cpu_prefill.py holds it to; the bound is test_gpu_prefill's."""
import numpy as np
import pytest
import torch

from oracle import fq_oracle as O
from tests.cases import to_dev, to_dev_half
from tests.test_gpu_prefill import ATOL, PrefillCase, _check, _turbo_case

pytestmark = pytest.mark.gpu

# (shape, (key groups, key-range splits), row blocks with empty slices)
FORMS = [
    (dict(Hq=6, Hkv=2, S=256, T=44), (4, 1), 0),                                     # 900 rows
    (dict(Hq=2, Hkv=2, S=256, T=1), (4, 1), 0),                                      # one row past 4 blocks of 64
    (dict(Hq=2, Hkv=2, S=1024, T=2, Sq=64, causal_offset=962), (4, 2), 0),           # one whole block, 9 stages
    (dict(Hq=6, Hkv=2, S=1536, T=54, Sq=90, causal_offset=1500), (4, 3), 0),
    (dict(Hq=64, Hkv=16, S=3072, T=18, Sq=90, causal_offset=3000), (2, 5), 0),
    (dict(Hq=64, Hkv=64, S=960, T=0, Sq=260, causal_offset=700), (2, 1), 0),
    (dict(Hq=64, Hkv=64, B=2, S=512, T=48, Sq=260, causal_offset=300), (1, 1), 0),
    (dict(Hq=6, Hkv=2, S=1536, T=54, Sq=300, causal_offset=0), (4, 1), 0),           # torch's is_causal over a longer cache
]
SPLIT_FORMS = [
    (dict(Hq=1, Hkv=1, S=3200, T=56, Sq=256, causal_offset=3000), (4, 6), 2),
    (dict(Hq=6, Hkv=2, S=2496, T=4, Sq=1000, causal_offset=1500), (2, 5), 3),
    (dict(Hq=12, Hkv=12, B=4, S=2496, T=31, Sq=142, causal_offset=2385), (1, 5), 0), # one row block
    (dict(Hq=24, Hkv=8, S=2176, T=24, Sq=700, causal_offset=1500), (1, 3), 0),
    (dict(Hq=3, Hkv=3, S=6912, T=1, Sq=2818, causal_offset=4095), (1, 7), 1),
]


@pytest.mark.parametrize("kw", [kw for kw, _, _ in FORMS])
def test_prefill_dense_forms(kw):
    _check(PrefillCase(17, **kw))


def _attention(Q, K, V, off):
    """Causal GQA attention in 64 bits, one head at a time."""
    q, k, v = (torch.from_numpy(np.ascontiguousarray(x)).double() for x in (Q, K, V))
    out = torch.empty_like(q)
    masked = torch.arange(k.shape[2])[None] > torch.arange(q.shape[2])[:, None] + off
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            kv = h // (q.shape[1] // k.shape[1])
            z = (q[b, h] @ k[b, kv].T / q.shape[3] ** 0.5).masked_fill_(masked, -torch.inf)
            out[b, h] = z.softmax(-1) @ v[b, kv]
    return out.numpy()


@pytest.mark.parametrize("bits", [4, 8, 3])
@pytest.mark.parametrize("kw", [kw for kw, _, _ in SPLIT_FORMS])
def test_prefill_split_forms(kw, bits):
    print(f"[prefill splits] bits={bits} {kw}", flush=True)
    if bits == 3:
        from flashquest_amd.kernel import flash_attn_prefill_turbo
        S = kw["S"]
        K, V, Q, planes = _turbo_case(23, **{k: v for k, v in kw.items() if k != "causal_offset"})
        dev = [to_dev(p) if i % 3 < 2 else to_dev_half(p, "bf16") for i, p in enumerate(planes)]
        out = flash_attn_prefill_turbo(to_dev_half(Q, "bf16"), *dev, to_dev_half(K[:, :, S:], "bf16"),
                                       to_dev_half(V[:, :, S:], "bf16"), page_size=64, causal_offset=kw["causal_offset"])
        Kf, Vf = (np.concatenate([O.dequant_turbo_bf16(*planes[i:i + 3]), X[:, :, S:]], axis=2)
                  for i, X in ((0, K), (3, V)))
    else:
        c = PrefillCase(23, bits=bits, **kw)
        out, Q = c.run(), c.Q
        Kf = np.concatenate([O.dequant_cache_bf16(c.kc, "K", c.ks, c.km, c.page, bits), c.Kt], axis=2)
        Vf = np.concatenate([O.dequant_cache_bf16(c.vc, "V", c.vs, c.vm, c.page, bits), c.Vt], axis=2)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all()
    err = float(np.abs(got - _attention(Q, Kf, Vf, kw["causal_offset"])).max())
    assert err < ATOL, err
