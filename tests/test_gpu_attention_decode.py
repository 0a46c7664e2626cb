"""GPU parity of the decode attention kernel (flash_dec_kernel): few queries
per KV head, the keys split over waves and workgroups.

Tolerance of the bf16 layers: normwise 2e-2 against the oracle's op sequence;
repeated runs are equal bit for bit (the splits merge in one order).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from rew_amd import eager as E
from rew_amd import nn
from rew_amd.eager import DType
from test_gpu_attention import _expand, _qkv, _run


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,D", [
    (1, 8, 4, 1, 128, 128),    # one tile per wave, two columns in use
    (1, 4, 4, 3, 1000, 128),   # one query head per KV head
    (2, 8, 2, 4, 129, 64),     # a last tile of one key
    (1, 32, 8, 8, 200, 128),   # every column in use
    (3, 6, 2, 1, 1000, 32),
    (16, 32, 8, 1, 300, 128),  # pairs beyond half of the CUs
    (40, 32, 16, 2, 192, 64),  # more pairs than CUs: no split
    (1, 8, 1, 4, 4097, 64),    # one pair over many workgroups
])
def test_decode_matches_oracle(gpu, oracle, causal, B, H, Hkv, Sq, Sk, D):
    q, k, v = _qkv(oracle, 77 + Sk + D, B, H, Hkv, Sq, Sk, D)
    g = H // Hkv
    qt, kt, vt = (E.fromHost(t, DType.BFLOAT16) for t in (q, k, v))

    def fn():
        return nn.scaledDotProductAttention(qt, _expand(kt, B, Hkv, g, Sk, D),
                                            _expand(vt, B, Hkv, g, Sk, D), causal=causal)

    got, names = _run(fn)
    assert any(n.startswith("flash_attn_dec") for n in names), names
    want = oracle.sdpa(q, k, v, 1 if causal else 0, mixed=True)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= 2e-2, err
    assert np.max(np.abs(got - want)) <= 1e-1 * np.max(np.abs(want))
    for _ in range(3):
        np.testing.assert_array_equal(_run(fn)[0], got)
