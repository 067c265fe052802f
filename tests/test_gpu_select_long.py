"""Selection past the in-kernel 512 pages at the edges of its register layouts
(64 C pages, C = 16 and 32), for every head count of a workgroup and both modes,
few groups and many: bit for bit against the oracle, and O and lse within the
decode bars."""
import numpy as np
import pytest
import torch

from oracle import fq_oracle as O
from tests.cases import Int4Case, decode_tol, max_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,nrep,mode,Hkv", [(513, 1, "per_q_head", 2), (1024, 3, "per_q_head", 1), (1025, 4, "per_q_head", 1),
                                             (2048, 2, "per_q_head", 1), (1023, 4, "per_kv_head_sum", 2),
                                             (2047, 3, "per_kv_head_sum", 1), (2049, 3, "per_q_head", 1), (600, 8, "per_q_head", 1)])
def test_long_selection(P, nrep, mode, Hkv):
    from flashquest_amd.eager.decode import quest_decode_int4
    c = Int4Case(seed=P, B=1, Hq=nrep * Hkv, Hkv=Hkv, S=64 * P - 9, D=64)
    kw = dict(retention=0.2, num_sinks=4, window_pages=2)
    o, lse, mask = quest_decode_int4(c.q_dev(), **c.device(), select_mode=mode, return_selection=True, **kw)
    o2, _ = quest_decode_int4(c.q_dev(), **c.device(), select_mode=mode, **kw)
    torch.cuda.synchronize()
    ref = O.decode_step(c.Q, c.kp, c.ks, c.km, c.vp, c.vs, c.vm, mode=mode, **kw)
    assert np.array_equal(mask.cpu().numpy(), ref["mask"])
    for x in (o, o2):
        assert max_err(x[:, :, 0], ref["O"]) <= decode_tol(ref["O"], "bf16")
    assert max_err(lse[:, :, 0], ref["lse"]) <= 1e-4
