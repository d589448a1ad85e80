"""GPU parity of the two-launch split-KV path: a row's workgroups counted and
summed by the last of them (up to two levels of 16), statistics joined in the
P.V launch, workgroups found in ragged lengths.  Oracle and gate as in
tests/common.py."""
import numpy as np
import pytest

import oracle
from tests.common import assert_pass, default_scale, last_plan, make_inputs, plan_kinds, plan_launch, to_dev

pytestmark = pytest.mark.gpu


def _ragged(B, max_len, seed):
    rng = np.random.default_rng(seed)
    lens = np.exp(rng.uniform(0, np.log(max_len), size=B)).astype(np.int32)
    edge = [max_len, 0, 1, 128, 129, 127, 256, 2048, 2049]
    lens[:min(B, len(edge))] = np.minimum(edge, max_len)[:min(B, len(edge))]
    return lens


def _call(q, k, v, cu, max_len, D, ws):
    import fmha_amd
    return fmha_amd.fmha_decode_splitkv(q, k, v, cu, max_len, softmax_scale=default_scale(D), workspace=ws)


def _workspace(B, Hq, Hkv, max_len, D, fill):
    import torch
    import fmha_amd
    ws = torch.empty(fmha_amd.splitkv_workspace_size(B, Hq, Hkv, max_len, D), dtype=torch.uint8, device="cuda")
    return ws.fill_(fill)


# (B, Hq, Hkv, D, max_len, rows per P.V workgroup or None for the planner's):
# one workgroup per row, 2, 16 and 17 (one level of sums and two), 40; one to
# five lane columns per query group (G = 1, 2, 4, 8, 16) and two tiles with
# the second half full (24, padded from 20); the wave's batch scan on one
# register, two, at its limit (256) and past it; rows of one wave.
CASES = [
    (3, 8, 8, 128, 200, None),
    (2, 16, 8, 128, 256, 128),
    (5, 32, 8, 128, 2048, 128),
    (9, 32, 8, 128, 2049, 128),
    (1, 8, 2, 64, 5120, 128),
    (4, 16, 2, 256, 2100, 128),
    (6, 32, 2, 128, 700, 128),
    (3, 20, 1, 128, 4200, 128),
    (2, 20, 1, 256, 600, None),
    (65, 2, 1, 64, 2100, 256),
    (70, 8, 1, 128, 2300, None),
    (256, 1, 1, 64, 700, 256),
    (257, 1, 1, 128, 300, 128),
    (30, 8, 8, 64, 64, None),
    (7, 48, 2, 256, 64, None),
    (40, 2, 1, 256, 33, None),
]


@pytest.mark.parametrize("B,Hq,Hkv,D,max_len,rows", CASES)
def test_ragged_rows(monkeypatch, B, Hq, Hkv, D, max_len, rows):
    """Ragged lengths (0, 1, the edges of a workgroup's rows, the maximum), a
    workspace full of NaN patterns, and the same bits a second time from one
    full of zeros, and through the same workspace again."""
    import torch
    if rows:
        monkeypatch.setenv("FMHA_DECODE_SPLIT_CHUNK", str(rows))
    monkeypatch.setenv("FMHA_DECODE_ONEPASS_REG", "0")
    monkeypatch.setenv("FMHA_DECODE_ONEPASS_MFMA", "0")
    lens = _ragged(B, max_len, B * 5 + max_len)
    q, k, v, cu = make_inputs(B, Hq, Hkv, D, lens, seed=B + D + Hq, std=0.5)
    dev = [to_dev(x) for x in (q, k, v)] + [torch.from_numpy(cu).cuda()]
    outs = []
    for fill in (0xFF, 0x00, None):
        if fill is not None:
            ws = _workspace(B, Hq, Hkv, max_len, D, fill)
        o = _call(*dev, max_len, D, ws)
        assert any(p.startswith("split") for p in plan_kinds()), plan_kinds()
        torch.cuda.synchronize()
        outs.append(o.view(torch.int16).cpu().numpy().view(np.uint16))
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
    r, slack = oracle.decode(q, k, v, cu, Hq, Hkv, D, default_scale(D), with_slack=True, max_seqlen=max_len)
    assert_pass(oracle.compare(outs[0].reshape(r.shape), r, slack), f"B={B} G={Hq // Hkv} D={D} max={max_len}")


def test_many_calls_same_bits():
    """200 calls through one workspace on one stream, with other work between
    them, and calls on two streams with a workspace each: always the same
    bits, whichever workgroup of a row finishes last."""
    import torch
    B, Hq, Hkv, D, max_len = 3, 32, 8, 128, 9000
    lens = np.array([9000, 4097, 700], np.int32)
    q, k, v, cu = make_inputs(B, Hq, Hkv, D, lens, seed=77, std=0.5)
    dev = [to_dev(x) for x in (q, k, v)] + [torch.from_numpy(cu).cuda()]
    ws = [_workspace(B, Hq, Hkv, max_len, D, 0xFF) for _ in range(2)]
    first = _call(*dev, max_len, D, ws[0]).clone()
    assert plan_launch("split")["launches"] == 2
    noise = torch.randn(1 << 20, device="cuda")
    for i in range(200):
        o = _call(*dev, max_len, D, ws[0])
        if i % 3 == 0:
            noise.mul_(1.0001)
        assert torch.equal(o.view(torch.int16), first.view(torch.int16)), i
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    for i in range(20):
        got = []
        for s, w in zip(streams, ws):
            with torch.cuda.stream(s):
                got.append(_call(*dev, max_len, D, w))
        torch.cuda.synchronize()
        for o in got:
            assert torch.equal(o.view(torch.int16), first.view(torch.int16)), i


# (layout, Hq, Hkv, D, max_len, lengths, parts): lengths far
# below the longest row allowed, for which the device takes shorter pieces than
# planned (one batch, a few, one register of lengths and more), and as long,
# for which it keeps them; head dims whole and by halves; empty and invalid
# batches.  -1 stands for max_len + 1.
CHOSEN = [
    ("packed", 32, 8, 128, 131072, [5000], 1),
    ("packed", 8, 8, 256, 60000, [3000], 2),
    ("paged16", 64, 8, 128, 32768, [9000, 0, 2049, -1, 700, 1], 1),
    ("strided", 8, 8, 64, 9000, [9000] + [400] * 11, 1),
    ("packed", 16, 2, 256, 16384, [6000, 0, 300, 16], 2),
    ("paged16", 8, 8, 256, 11516, [4000, -1, 0, 900, 257] + [100] * 5, 1),
    ("strided", 2, 2, 256, 4096, [3000] + [150] * 43, 2),
    ("paged1", 8, 1, 256, 8192, [5000, 600] + [250] * 18, 2),
    ("packed", 1, 1, 64, 8000, [8000] + [300] * 69, 1),
    ("packed", 8, 8, 64, 2233, [2233] * 57, 1),
    ("paged16", 8, 8, 256, 4000, [4000] * 10 + [3500] * 12, 1),
]


@pytest.mark.parametrize("layout,Hq,Hkv,D,max_len,lens,parts", CHOSEN)
def test_device_chosen_pieces(monkeypatch, layout, Hq, Hkv, D, max_len, lens, parts):
    """What the device makes of the lengths, with a workspace of exactly the
    size asked for between guard bytes, which stay."""
    import torch
    import fmha_amd
    monkeypatch.setenv("FMHA_DECODE_ONEPASS_REG", "0")
    monkeypatch.setenv("FMHA_DECODE_ONEPASS_MFMA", "0")
    B = len(lens)
    invalid = [b for b, n in enumerate(lens) if n < 0]
    said = np.array([max_len + 1 if n < 0 else n for n in lens], np.int32)
    # An invalid batch's rows are not read: packed caches have none of it here.
    held = np.array([0 if n < 0 else n for n in lens], np.int32)
    assert layout != "packed" or not invalid
    q, k, v, cu = make_inputs(B, Hq, Hkv, D, held, seed=B + D + Hq + max_len, std=0.5)
    need, guard = fmha_amd.splitkv_workspace_size(B, Hq, Hkv, max_len, D), 4096
    room = torch.full((guard + need + guard,), 0xA5, dtype=torch.uint8, device="cuda")
    ws = room[guard:guard + need]
    ws.fill_(0xFF)
    scale = default_scale(D)
    ln = torch.from_numpy(said).cuda()
    if layout == "packed":
        call = lambda: _call(to_dev(q), to_dev(k), to_dev(v), torch.from_numpy(cu).cuda(), max_len, D, ws)  # noqa: E731
    elif layout == "strided":
        kc, vc = (torch.zeros(B, max_len, Hkv, D, dtype=torch.int16) for _ in range(2))
        for b in range(B):
            kc[b, :held[b]] = torch.from_numpy(k[cu[b]:cu[b + 1]].view(np.int16))
            vc[b, :held[b]] = torch.from_numpy(v[cu[b]:cu[b + 1]].view(np.int16))
        kc, vc = (x.cuda().view(torch.bfloat16) for x in (kc, vc))
        call = lambda: fmha_amd.fmha_decode_strided(to_dev(q), kc, vc, ln, softmax_scale=scale, workspace=ws)  # noqa: E731
    else:
        page = int(layout[5:])
        used = [(int(n) + page - 1) // page for n in held]
        perm = np.random.default_rng(3).permutation(sum(used)).astype(np.int32)
        table = np.full((B, (max_len + page - 1) // page), -1, np.int32)
        slots = np.zeros(len(k), np.int64)
        at = 0
        for b in range(B):
            table[b, :used[b]] = perm[at:at + used[b]]
            at += used[b]
            j = np.arange(held[b])
            slots[cu[b]:cu[b + 1]] = table[b, j // page].astype(np.int64) * page + j % page
        kc, vc = (np.zeros((sum(used) * page, Hkv, D), np.uint16) for _ in range(2))
        kc[slots], vc[slots] = k, v
        kc, vc = (to_dev(x.reshape(-1, page, Hkv, D)) for x in (kc, vc))
        bt = torch.from_numpy(table).cuda()
        call = lambda: fmha_amd.fmha_decode_paged(to_dev(q), kc, vc, bt, ln, softmax_scale=scale,  # noqa: E731
                                                  max_seqlen_kv=max_len, workspace=ws)
    first = call()
    split = [f for kind, f in last_plan() if kind.startswith("split")]
    assert len(split) == 1 and split[0]["pv_parts"] == parts, split
    assert split[0]["pv_rows"] > split[0]["pv_rows_least"] == 256, split  # the device has a choice
    second = call()
    torch.cuda.synchronize()
    assert bool((room[:guard] == 0xA5).all()) and bool((room[guard + need:] == 0xA5).all())
    bits = first.view(torch.int16).cpu().numpy().view(np.uint16)
    assert np.array_equal(bits, second.view(torch.int16).cpu().numpy().view(np.uint16))
    r, slack = oracle.decode(q, k, v, cu, Hq, Hkv, D, scale, with_slack=True, max_seqlen=max_len)
    bits = bits.reshape(r.shape)
    assert np.all(np.isnan(oracle.f16_to_f32(bits[invalid])))
    ok = [b for b in range(B) if b not in invalid]
    assert_pass(oracle.compare(bits[ok], r[ok], slack[ok]), f"{layout} B={B} G={Hq // Hkv} D={D} max={max_len}")


def test_longest_rows_allowed():
    """The longest rows that a batch's scores allow (below 2^30 bytes), of
    which few are there: accepted, the row's pieces counted in 131072 places;
    16 rows more are refused."""
    import torch
    import fmha_amd
    Hq, D, n, page = 8, 256, 700, 64
    max_len = 2 ** 25 - 16
    lens = np.array([n], np.int32)
    q, k, v, cu = make_inputs(1, Hq, Hq, D, lens, seed=9, std=0.5)
    used = (n + page - 1) // page
    kc, vc = (np.zeros((used * page, Hq, D), np.uint16) for _ in range(2))
    kc[:n], vc[:n] = k, v
    table = torch.full((1, (max_len + 16 + page - 1) // page), -1, dtype=torch.int32, device="cuda")
    table[0, :used] = torch.arange(used, dtype=torch.int32)
    args = (to_dev(q), *(to_dev(x.reshape(-1, page, Hq, D)) for x in (kc, vc)), table, torch.from_numpy(lens).cuda())
    o = fmha_amd.fmha_decode_paged(*args, softmax_scale=default_scale(D), max_seqlen_kv=max_len)
    torch.cuda.synchronize()
    r, slack = oracle.decode(q, k, v, cu, Hq, Hq, D, default_scale(D), with_slack=True, max_seqlen=n)
    bits = o.view(torch.int16).cpu().numpy().view(np.uint16)
    assert_pass(oracle.compare(bits.reshape(r.shape), r, slack), "longest rows")
    with pytest.raises(fmha_amd.FmhaDecodeError, match="too large"):
        fmha_amd.fmha_decode_paged(*args, softmax_scale=default_scale(D), max_seqlen_kv=max_len + 16)


@pytest.mark.parametrize("page_size", [1, 16, 64])
@pytest.mark.parametrize("Hq,Hkv,D", [(8, 8, 128), (16, 2, 64), (32, 1, 128), (4, 2, 256)])
def test_paged_ragged_rows(monkeypatch, page_size, Hq, Hkv, D):
    """The same over paged caches: rows in scattered pages, a negative entry
    past a batch's rows (not read), one among them (NaN for that batch)."""
    import torch
    import fmha_amd
    monkeypatch.setenv("FMHA_DECODE_SPLIT_CHUNK", "128")
    B, max_len = 6, 1000
    lens = np.array([1000, 0, 1, 513, 130, 64], np.int32)
    q, k, v, cu = make_inputs(B, Hq, Hkv, D, lens, seed=page_size + D + Hq, std=0.5)
    cols = (max_len + page_size - 1) // page_size
    used = [(int(n) + page_size - 1) // page_size for n in lens]
    perm = np.random.default_rng(3).permutation(sum(used)).astype(np.int32)
    table = np.full((B, cols), -1, np.int32)
    kc = np.zeros((sum(used), page_size, Hkv, D), np.uint16)
    vc = np.zeros_like(kc)
    at = 0
    for b in range(B):
        table[b, :used[b]] = perm[at:at + used[b]]
        at += used[b]
        for j in range(int(lens[b])):
            kc[table[b, j // page_size], j % page_size] = k[cu[b] + j]
            vc[table[b, j // page_size], j % page_size] = v[cu[b] + j]
    # an empty batch's first entry is looked up, never followed
    bt = torch.from_numpy(table).cuda()
    args = (to_dev(q), to_dev(kc), to_dev(vc))
    ln = torch.from_numpy(lens).cuda()
    o = fmha_amd.fmha_decode_paged(*args, bt, ln, softmax_scale=default_scale(D), max_seqlen_kv=max_len)
    assert any(p.startswith("split") for p in plan_kinds()), plan_kinds()
    torch.cuda.synchronize()
    bits = o.view(torch.int16).cpu().numpy().view(np.uint16)
    r, slack = oracle.decode(q, k, v, cu, Hq, Hkv, D, default_scale(D), with_slack=True, max_seqlen=max_len)
    assert_pass(oracle.compare(bits.reshape(r.shape), r, slack), f"paged{page_size} Hq={Hq} D={D}")
    table[3, used[3] - 1] = -1
    o2 = fmha_amd.fmha_decode_paged(*args, torch.from_numpy(table).cuda(), ln, softmax_scale=default_scale(D),
                                    max_seqlen_kv=max_len)
    torch.cuda.synchronize()
    f = oracle.f16_to_f32(o2.view(torch.int16).cpu().numpy().view(np.uint16)).reshape(B, -1)
    assert np.all(np.isnan(f[3])) and np.all(np.isfinite(np.delete(f, 3, axis=0)))
