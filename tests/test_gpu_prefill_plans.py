"""The dense prefill's forms (key groups per workgroup 1 / 2 / 4, with and
without key-range splits) against the CPU oracle: row counts around the 64-,
128- and 256-row blocks, key counts around the 128-key stages, whole prompts and
chunks over a cache.  The sizes below take each form (csrc/prefill.hip,
dense_plan); the bound is test_gpu_prefill's."""
import pytest

from tests.test_gpu_prefill import PrefillCase, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [
    dict(Hq=6, Hkv=2, S=256, T=44),                                        # 4 key groups: 900 rows
    dict(Hq=2, Hkv=2, S=256, T=1),                                         # one row past 4 blocks of 64
    dict(Hq=2, Hkv=2, S=1024, T=2, Sq=64, causal_offset=962),              # one whole block, 9 stages
    dict(Hq=6, Hkv=2, S=1536, T=54, Sq=90, causal_offset=1500),            # 4 key groups x 3 splits
    dict(Hq=64, Hkv=16, S=3072, T=18, Sq=90, causal_offset=3000),          # 2 key groups x 5 splits
    dict(Hq=64, Hkv=64, S=960, T=0, Sq=260, causal_offset=700),            # 2 key groups, one split
    dict(Hq=64, Hkv=64, B=2, S=512, T=48, Sq=260, causal_offset=300),      # 1 key group, one split
    dict(Hq=6, Hkv=2, S=1536, T=54, Sq=300, causal_offset=0),              # torch's is_causal over a longer cache
])
def test_prefill_dense_forms(kw):
    _check(PrefillCase(17, **kw))
