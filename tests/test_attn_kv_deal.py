"""Pairs of q blocks whose kv blocks are dealt to several programs one by one (SYN_ATTN_SPLIT_DEAL): the plan (host), which
tables keep their parts in wave order instead, and launches at the sizes where the deal goes round differently."""

import pytest
import torch

from oracle import numerics
from syncopate_amd.computation.attn.kv_split import BLOCK, KvSplit, plan_kv_deal, plan_kv_split


def _tables(Z, H, Sq, lengths, signals):
    offsets, sizes, cums, lo = [], [], [], 0
    for i, n in enumerate(lengths):
        offsets.append([0, 0, 0, lo])
        sizes.append([Z, H, Sq, n])
        cums.append((i + 1) * Z * H * Sq)
        lo += n
    return offsets, sizes, cums, signals


def test_plans_of_tables_that_wait():
    plan = lambda Z, H, Sq, lengths, signals: plan_kv_deal(*_tables(Z, H, Sq, lengths, signals), units=256)
    gated = lambda waves: [-1] + list(range(waves - 1))
    # the last chunk's blocks are shared by seven parts; 32 units stay free for the kernels that raise the flags
    assert plan(1, 8, 1024, [1024] * 8, gated(8)) == KvSplit(True, 32, 7, 10)
    for heads in range(1, 66):
        for sq in (256, 1024, 3072):
            got = plan(1, heads, sq, [1024] * 8, gated(8))
            assert got is None or (got.programs <= 224 and got.chain)
    # short launches, which the host bounds; enough tiles to fill the device; q blocks that do not pair up or differ
    assert plan(1, 2, 512, [128] * 2, gated(2)) is None
    assert plan(1, 32, 4096, [4096] * 8, gated(8)) is None
    assert plan(1, 8, 1152, [1024] * 8, gated(8)) is None
    assert plan_kv_deal([[0, 0, 0, 0], [0, 0, 256, 0]], [[1, 2, 256, 4096]] * 2, [512, 1024], [-1, 0], units=256) is None
    assert plan_kv_deal([[0, 0, 0, 0]], [[1, 1, 256, 128]], [0], [-1], units=256) is None


@pytest.mark.parametrize("H,Sq,lengths,always,split", [
    (49, 2816, [18 * 128] * 8, True, (539, 2)),       # more parts than slots, one of each pair's in registers
    (50, 3072, [30 * 128] * 4, True, (600, 2)),
    (8, 1024, [1024] * 8, True, (32, 8)),
    (8, 1536, [1536] * 4, False, (48, 4)),            # the template's own call
])
def test_cut_in_wave_order(H, Sq, lengths, always, split):
    """Tables whose parts have always been added in 32 bits: the parts in wave order that they had."""
    got = plan_kv_split(*_tables(1, H, Sq, lengths, [-1] * len(lengths)), causal=False, producer=False, units=256, always=always)
    assert (got.pairs, got.parts) == split and got.blocks == -(-sum(lengths) // (128 * split[1]))


def _parts_by_hand(q, k, v, scale, parts):
    """[rows, 128] of one head: each part's blocks in the order given, probabilities rounded against the maximum so far, and the
    parts' sums added neighbour to neighbour."""
    sums = []
    for blocks in parts:
        m, l, o = torch.full((len(q), 1), -3e38), torch.zeros(len(q), 1), torch.zeros(len(q), 128)
        for b in blocks:
            s = q.float() @ k[b * BLOCK:(b + 1) * BLOCK].float().T * (scale * 1.4426950408889634)
            top = torch.maximum(m, s.max(dim=1, keepdim=True).values)
            p = torch.exp2(s - top)
            l = l * torch.exp2(m - top) + p.sum(dim=1, keepdim=True)
            o = o * torch.exp2(m - top) + p.to(v.dtype).float() @ v[b * BLOCK:(b + 1) * BLOCK].float()
            m = top
        sums.append((m, l, o))
    while len(sums) > 1:
        pairs = [sums[i:i + 2] for i in range(0, len(sums), 2)]
        sums = [pair[0] if len(pair) == 1 else _add(*pair) for pair in pairs]
    return (sums[0][2] / sums[0][1]).to(q.dtype)


def _add(a, b):
    top = torch.maximum(a[0], b[0])
    wa, wb = torch.exp2(a[0] - top), torch.exp2(b[0] - top)
    return top, a[1] * wa + b[1] * wb, a[2] * wa + b[2] * wb


@pytest.mark.gpu
@pytest.mark.parametrize("lengths,parts,form", [([128 * 12], 4, "explicit"), ([128 * 5, 128 * 3, 128 * 7], 3, "auto"), ([128 * 9], 7, "auto")])
def test_parts_in_wave_order_keep_their_results(hip, monkeypatch, lengths, parts, form):
    """A table that `plan_kv_split` cuts gives the results of parts that are runs of blocks, whichever program adds them."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward

    offsets, sizes, cums, signals = _tables(1, 1, 256, lengths, [-1] * len(lengths))
    total = sum(lengths) // BLOCK
    g = torch.Generator().manual_seed(11)
    q, k, v = (torch.randn(1, 1, s, 128, generator=g).bfloat16() for s in (256, total * BLOCK, total * BLOCK))
    each = -(-total // parts)
    monkeypatch.setattr("syncopate_amd.computation.attn.template.plan_kv_split", lambda *args, **kwargs: KvSplit(True, 1, parts, each))
    o = attention_forward(q.cuda(), k.cuda(), v.cuda(), 128 ** -0.5, wave_offsets=offsets, wave_sizes=sizes, cum_wave_sizes=cums,
                          signal_offsets=signals, signal_ptr=torch.ones(1, dtype=torch.int64, device="cuda"), cum_tiles=cums[-1],
                          form=form)
    check_status()
    real = -(-total // each)
    runs = [range(total * i // real, total * (i + 1) // real) for i in range(real)]
    want = _parts_by_hand(q[0, 0], k[0, 0], v[0, 0], 128 ** -0.5, runs)
    # The same roundings of every probability, sums in 32 bits in another order: scores 2^-21 apart move one probability in 1000
    # to the other side of a rounding and with it one result in 100 or 200.  Blocks met in another order round most of them
    # anew and a third of the results.
    assert (o[0, 0].cpu() == want).float().mean() >= 0.97


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
@pytest.mark.parametrize("Z,H,Sq,lengths,parts", [
    (1, 1, 256, [128], 3),                       # fewer blocks than parts: two parts of nothing
    (1, 3, 256, [128 * 5, 128, 128 * 9], 4),     # waves that some parts have no block of
    (2, 1, 512, [128] * 70, 16),                 # more waves than are looked at at a time
    (1, 9, 1024, [128 * 3] * 4, 7),              # programs dealt to the XCDs unevenly
    (1, 75, 1024, [128, 256], 2),                # more programs than compute units
])
def test_dealt_blocks_add_up(hip, monkeypatch, Z, H, Sq, lengths, parts, layout):
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward

    waves, Skv = len(lengths), sum(lengths)
    # every other wave is behind a flag, and the table ends in a row of padding
    offsets, sizes, cums, _ = _tables(Z, H, Sq, lengths, None)
    signals = [i if i % 2 else -1 for i in range(waves)]
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(Z, H, s, 128, generator=g).bfloat16() for s in (Sq, Skv, Skv))
    lay = lambda t: t if layout == "bhsd" else t.permute(0, 2, 1, 3).contiguous()
    monkeypatch.setattr("syncopate_amd.computation.attn.template.plan_kv_split", lambda *args, **kwargs: None)
    monkeypatch.setattr("syncopate_amd.computation.attn.template.plan_kv_deal",
                        lambda *args, **kwargs: KvSplit(True, Z * H * Sq // 256, parts, -(-Skv // (BLOCK * parts))))
    flags = torch.ones(waves, dtype=torch.int64, device="cuda")
    o, lse = attention_forward(lay(q).cuda(), lay(k).cuda(), lay(v).cuda(), 128 ** -0.5, wave_offsets=offsets + [[0] * 4],
                               wave_sizes=sizes + [[0] * 4], cum_wave_sizes=cums + [0], signal_offsets=signals + [0],
                               signal_ptr=flags, cum_tiles=cums[-1], layout=layout, return_lse=True)
    check_status()
    want = numerics.sdpa_fp32(q, k, v, 128 ** -0.5)
    # one rounding of the result and one of the probabilities, 2^-9 each, relative to the largest value; three times that
    assert ((o if layout == "bhsd" else o.permute(0, 2, 1, 3)).float().cpu() - want).abs().max() <= \
        1.2e-2 * want.abs().max()
    s = (q.float() @ k.float().transpose(-1, -2)) * 128 ** -0.5
    assert (lse.cpu() - torch.logsumexp(s, dim=-1) / 0.6931471805599453).abs().max().item() <= 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("trusted", [True, False])
def test_chunks_that_come_late(hip, trusted):
    """A table that the launcher deals by itself: flags raised one after the other and out of order, by kernels that are
    launched behind it; the same bits as with every flag up."""
    from syncopate_amd import _lib
    from syncopate_amd.communication.comm_runtime.streams import pick_side_streams
    from syncopate_amd.computation._launch import check_status, compute_units, trust_flags
    from syncopate_amd.computation.attn import attention_forward

    H, Sq, chunk, chunks = 8, 1024, 1024, 8
    offsets, sizes, cums, signals = _tables(1, H, Sq, [chunk] * chunks, [-1] + list(range(chunks - 1)))
    assert plan_kv_deal(offsets, sizes, cums, signals, units=compute_units(0))
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (torch.randn(1, H, s, 128, device="cuda", generator=g).bfloat16() for s in (Sq, chunk * chunks, chunk * chunks))
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    tables = dict(wave_offsets=table(offsets), wave_sizes=table(sizes), cum_wave_sizes=table(cums), signal_offsets=table(signals),
                  cum_tiles=cums[-1])
    flags = torch.ones(chunks, dtype=torch.int64, device="cuda")
    if trusted:
        trust_flags(flags)
    resident = attention_forward(q, k, v, 128 ** -0.5, signal_ptr=flags, **tables)
    lib, side = _lib.load(), pick_side_streams(1)[0]
    for first in (0, 3):
        flags.zero_()
        torch.cuda.synchronize()
        o = attention_forward(q, k, v, 128 ** -0.5, signal_ptr=flags, **tables)
        for i in range(chunks - 1):
            _lib.check("syn_delay_us", lib.syn_delay_us(20, _lib.stream_handle(side)))
            _lib.check("syn_flag_set", lib.syn_flag_set(flags.data_ptr() + 8 * ((first + 2 * i) % 7), 1, _lib.stream_handle(side)))
        check_status()
        assert torch.equal(o, resident)


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["fewer pairs", "other rows", "flag that stays down", "flag of the last wave"])
def test_refused_launch_writes_nothing(hip, monkeypatch, what):
    """A table that is not the one the launch was planned for, or a flag that does not come: the first kernel says so, and the second
    leaves the result as it was."""
    from syncopate_amd import _lib
    from syncopate_amd.computation._launch import FlagWaitTimeout, check_status
    from syncopate_amd.computation.attn import attention_forward, template

    H, parts = 2, 3
    offsets, sizes, cums, signals = _tables(1, H, 256, [512, 512], [-1, -1])
    flags = torch.ones(2, dtype=torch.int64, device="cuda")
    pairs, timeout = H, {}
    if what == "fewer pairs":
        pairs = 2 * H
    elif what == "other rows":
        offsets[1][2] = 256
    else:
        signals = [0, 1] if what == "flag that stays down" else [-1, 1]
        flags[signals[0] if signals[0] >= 0 else 1] = 0
        timeout = dict(spin_timeout_us=2000)
    monkeypatch.setattr(template, "plan_kv_split", lambda *args, **kwargs: None)
    monkeypatch.setattr(template, "plan_kv_deal", lambda *args, **kwargs: KvSplit(True, pairs, parts, -(-8 // parts)))
    monkeypatch.setattr(template, "already_checked", lambda *args: True)
    g = torch.Generator(device="cuda").manual_seed(2)
    q, k, v = (torch.randn(1, H, s, 128, device="cuda", generator=g).bfloat16() for s in (512, 1024, 1024))
    # results of another launch where the allocator will put the parts
    stale = torch.full((pairs * parts * _lib.SYN_ATTN_SPLIT_SLOT_BYTES,), 1, dtype=torch.uint8, device="cuda")
    del stale
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    out = torch.full_like(q, 7.0)
    attention_forward(q, k, v, 0.1, wave_offsets=table(offsets), wave_sizes=table(sizes), cum_wave_sizes=table(cums),
                      signal_offsets=table(signals), signal_ptr=flags, cum_tiles=cums[-1], out=out, **timeout)
    with pytest.raises(FlagWaitTimeout if timeout else RuntimeError, match="timed out" if timeout else rf"\[{_lib.SYN_STATUS_BAD_CHAIN}, "):
        check_status()
    assert bool((out == 7.0).all())
