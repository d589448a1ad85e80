"""GPU parity of ragged batches on the register single pass: a row's tiles
shared evenly among its waves whatever its length, and the batches taken
longest row first.  Oracle and gate as in tests/common.py."""
import numpy as np
import pytest

import oracle
from tests.common import assert_pass, default_scale, make_inputs, plan_launch, to_dev

pytestmark = pytest.mark.gpu


def _run(q, k, v, cu, max_len, D):
    import torch
    import fmha_amd
    o = fmha_amd.fmha_decode_splitkv(to_dev(q), to_dev(k), to_dev(v), torch.from_numpy(cu).cuda(), max_len,
                                     softmax_scale=default_scale(D))
    torch.cuda.synchronize()
    return o.view(torch.int16).cpu().numpy().view(np.uint16)


# (B, Hq, Hkv, D, max_len): more waves than the CUs hold at once, with batch
# counts in one ordering lane register, one past it, at the ordering's limit
# (256) and one past that (batch order); 8, 16 and 32 tiles per wave.
ORDER_CASES = [
    (64, 32, 8, 128, 4096),
    (65, 16, 8, 128, 2100),
    (200, 16, 4, 64, 900),
    (256, 64, 8, 128, 500),
    (257, 64, 8, 128, 300),
]


@pytest.mark.parametrize("B,Hq,Hkv,D,max_len", ORDER_CASES)
def test_longest_rows_first(B, Hq, Hkv, D, max_len):
    """Lengths over the whole range with ties (many batches of one block
    count), empty rows, rows on the edges of a round's tiles, an invalid
    length (NaN for its batch only): every batch served exactly once."""
    rng = np.random.default_rng(B + max_len)
    seqlens = np.exp(rng.uniform(np.log(1), np.log(max_len), size=B)).astype(np.int32)
    seqlens[:8] = [max_len, 0, 1, 64, 65, 16, 17, 63]
    seqlens[B // 2:B // 2 + 6] = 33  # ties
    seqlens[-1] = max_len
    q, k, v, cu = make_inputs(B, Hq, Hkv, D, seqlens, seed=B * 3 + D, std=0.5)
    o = _run(q, k, v, cu, max_len, D)
    assert plan_launch("onepass_matrix_core_regs")["blocks"] == (max_len + 15) // 16
    r, slack = oracle.decode(q, k, v, cu, Hq, Hkv, D, default_scale(D), with_slack=True, max_seqlen=max_len)
    assert_pass(oracle.compare(o.reshape(r.shape), r, slack), f"ragged B={B} D={D} max={max_len}")
    # one row fewer allowed: the batches of max_len rows turn NaN, the rest keep their bits
    o2 = _run(q, k, v, cu, max_len - 1, D).reshape(B, -1)
    f2 = oracle.f16_to_f32(o2)
    full = seqlens == max_len
    assert np.all(np.isnan(f2[full])) and np.array_equal(o2[~full], o.reshape(B, -1)[~full])


def test_equal_lengths_keep_batch_order():
    """One length for every batch: no reordering, oracle parity."""
    B, Hq, Hkv, D, S = 70, 32, 8, 128, 2049
    q, k, v, cu = make_inputs(B, Hq, Hkv, D, np.full(B, S, np.int32), seed=5, std=0.5)
    o = _run(q, k, v, cu, S, D)
    r, slack = oracle.decode(q, k, v, cu, Hq, Hkv, D, default_scale(D), with_slack=True, max_seqlen=S)
    assert_pass(oracle.compare(o.reshape(r.shape), r, slack), "equal lengths")
