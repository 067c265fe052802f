"""The page quantisers' codes where their arithmetic can go wrong, bit for bit
against the oracle: quotients at and beside ties, scales from the 1e-6 floor to
1e38 (past the reciprocal form's range, in single channels and everywhere), pages
and token groups that end early, both head sizes and code widths, and code planes
whose alignment sends the call to the general kernel."""
import numpy as np
import pytest
import torch

from oracle import fq_oracle as O
from tests.cases import TORCH_HALF, to_dev

pytestmark = pytest.mark.gpu

TORCH = dict(TORCH_HALF, f32=torch.float32)


def _values(kind, rng, B, H, S, D, dtype):
    rnd = O.rounder(dtype)
    x = rng.standard_normal((B, H, S, D)).astype(np.float32)
    if kind == "ties":          # whole and half steps of power-of-two scales
        x = rng.integers(0, 31, (B, H, S, D)).astype(np.float32) / 2
        x[:, :, ::7] = 0.0
        x[:, :, 3::7] = 15.0
    elif kind == "wide":        # beyond 1e30 everywhere, and in a few channels / tokens only
        x = x * np.where(rng.random((B, H, 1, D)) < 0.1, 3e37, 1.0).astype(np.float32)
        x[:, :, ::5] *= np.float32(1e-3)
        x = np.clip(x, -1.6e38, 1.6e38)
    elif kind == "tiny":        # ranges below the scale floor
        x = x * np.float32(1e-7)
        x[..., 3] = 2.0
    return rnd(x)


def _bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


@pytest.mark.parametrize("kind", ["normal", "ties", "wide", "tiny"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("dtype,D,S", [("bf16", 128, 64 * 3), ("bf16", 64, 64 * 2 + 1), ("f32", 128, 63), ("f16", 64, 200)])
def test_codes(kind, bits, dtype, D, S):
    from flashquest_amd.kernel import quantize_k, quantize_k_int4, quantize_v, quantize_v_int4
    if dtype == "f16" and kind == "wide":
        pytest.skip("1e37 is not an fp16 value")
    rng = np.random.default_rng(S + D + bits)
    X = _values(kind, rng, 2, 3, S, D, dtype)
    dev = to_dev(X).to(TORCH[dtype])
    if bits == 4:
        want = [(O.quantize_k_int4(X, 64, dtype, "bf16"), quantize_k_int4(dev, 64)),
                (O.quantize_v_int4(X, None, "bf16"), quantize_v_int4(dev))]
        if D == 128:
            want.append((O.quantize_v_int4(X, 32, "bf16"), quantize_v_int4(dev, v_group=32)))
    else:
        want = [(O.quantize_k_int8(X, 64, dtype, "bf16"), quantize_k(dev, 64)),
                (O.quantize_v_int8(X, "bf16"), quantize_v(dev))]
    for (codes, scale, mn), (c, s, m) in want:
        assert np.array_equal(c.cpu().numpy(), codes)
        assert np.array_equal(_bits(s), O.to_bits(scale, "bf16"))
        assert np.array_equal(m.float().cpu().numpy(), mn)      # by value: numpy's minimum of 0 and -0 is either


@pytest.mark.parametrize("bits", [4, 8])
def test_code_planes_of_any_alignment(bits):
    """Planes 2 bytes off a 4- or 8-byte boundary take the general kernels: the same codes."""
    from flashquest_amd.kernel import quantize_k, quantize_k_int4, quantize_v, quantize_v_int4
    kq, vq = (quantize_k_int4, quantize_v_int4) if bits == 4 else (quantize_k, quantize_v)
    rng = np.random.default_rng(bits)
    dev = to_dev(_values("normal", rng, 1, 2, 130, 128, "bf16")).to(torch.bfloat16)
    for q, args in ((kq, (64,)), (vq, ())):
        c, s, m = q(dev, *args)
        n = c.numel()
        off = torch.zeros(n + 8, dtype=torch.uint8, device="cuda")[2:2 + n].view(c.shape)
        s2, m2 = torch.zeros_like(s), torch.zeros_like(m)
        q(dev, *args, out=(off, s2, m2))
        assert torch.equal(off, c) and torch.equal(s2, s) and torch.equal(m2, m)
