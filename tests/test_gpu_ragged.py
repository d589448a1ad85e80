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
# counts of one ordering group (up to 64), one past it, of four full groups
# (256) and one past that; 8, 16 and 32 tiles per wave.
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


# (layout, B, Hq, Hkv, D, max_len): one wave per unit, more units than start
# at once: 16- and 8-row sub-blocks, G = 1 to 8, ordering groups of unequal
# sizes (B not a multiple of their count), one of them a single batch over.
ONEPASS_CASES = [
    ("packed", 1100, 32, 8, 128, 100),
    ("packed", 2111, 64, 8, 64, 40),
    ("packed", 321, 32, 32, 128, 90),
    ("packed", 700, 32, 16, 256, 50),
    ("bhsd", 1089, 32, 8, 128, 70),
    (16, 1100, 64, 8, 128, 100),
    (16, 300, 32, 32, 128, 100),
    (1, 1090, 32, 8, 128, 40),
    (1, 300, 32, 32, 128, 40),
]


@pytest.mark.parametrize("layout,B,Hq,Hkv,D,max_len", ONEPASS_CASES)
def test_one_wave_rows_longest_first(layout, B, Hq, Hkv, D, max_len):
    """Rows of one wave, longest first: lengths over the whole range with
    ties, empty rows and the edges of one, two and three sub-blocks (a last
    one that stands alone is neither refilled nor followed)."""
    import torch
    import fmha_amd
    rng = np.random.default_rng(B + max_len)
    seqlens = np.exp(rng.uniform(0, np.log(max_len), size=B)).astype(np.int32)
    edges = np.minimum([max_len, 0, 1, 2, 7, 8, 9, 15, 16, 17, 24, 25, 31, 32, 33, 47, 48, 49], max_len)
    seqlens[:len(edges)] = edges
    seqlens[B // 2:B // 2 + 70] = 33
    seqlens[-1] = max_len
    q, k, v, cu = make_inputs(B, Hq, Hkv, D, seqlens, seed=B * 3 + D, std=0.5)
    qt, kt, vt = to_dev(q), to_dev(k), to_dev(v)
    lens = torch.from_numpy(seqlens).cuda()
    scale = default_scale(D)
    batch = torch.repeat_interleave(torch.arange(B), torch.from_numpy(seqlens).long())
    row = torch.arange(len(batch)) - torch.from_numpy(cu[:-1]).long()[batch]

    def run(limit):
        if layout == "packed":
            return fmha_amd.fmha_decode_splitkv(qt, kt, vt, torch.from_numpy(cu).cuda(), limit, softmax_scale=scale)
        if layout == "bhsd":
            pools = []
            for t in (kt, vt):
                p = torch.full((B, Hkv, limit, D), float("nan"), dtype=torch.bfloat16, device="cuda")
                keep = row < limit
                p[batch[keep].cuda(), :, row[keep].cuda()] = t.view(-1, Hkv, D)[keep.cuda()]
                pools.append(p.transpose(1, 2))
            return fmha_amd.fmha_decode_strided(qt.view(B, Hq, D), *pools, lens, softmax_scale=scale)
        width = (max_len + layout - 1) // layout
        used = (torch.from_numpy(seqlens).long() + layout - 1) // layout
        table = torch.full((B, width), -1, dtype=torch.int32)
        there = torch.arange(width)[None, :] < used[:, None]
        table[there] = torch.randperm(int(used.sum()), generator=torch.Generator().manual_seed(B)).to(torch.int32)
        slot = (table[batch, row // layout].long() * layout + row % layout).cuda()
        pools = []
        for t in (kt, vt):
            p = torch.full((int(used.sum()) * layout, Hkv, D), float("nan"), dtype=torch.bfloat16, device="cuda")
            p[slot] = t.view(-1, Hkv, D)
            pools.append(p.view(-1, layout, Hkv, D))
        return fmha_amd.fmha_decode_paged(qt.view(B, Hq, D), *pools, table.cuda(), lens, max_seqlen_kv=limit,
                                          softmax_scale=scale)

    def bits(o):
        torch.cuda.synchronize()
        return o.view(torch.int16).cpu().numpy().view(np.uint16).reshape(B, -1)

    o = bits(run(max_len))
    assert plan_launch("onepass")["blocks"] == (max_len + 15) // 16
    r, slack = oracle.decode(q, k, v, cu, Hq, Hkv, D, scale, with_slack=True, max_seqlen=max_len)
    assert_pass(oracle.compare(o.reshape(r.shape), r, slack), f"one wave per row, {layout} B={B} D={D} max={max_len}")
    # one row fewer allowed: the batches of max_len rows turn NaN, the rest keep their bits
    o2 = bits(run(max_len - 1))
    full = seqlens == max_len
    assert np.all(np.isnan(oracle.f16_to_f32(o2)[full])) and np.array_equal(o2[~full], o[~full])
