"""Attention whose pairs of q blocks are cut into parts along kv: the plan (host), and the launches against the fp32
reference at the sizes where the cuts fall differently."""

import pytest
import torch

from oracle import numerics
from syncopate_amd.computation.attn.kv_split import BLOCK, KvSplit, plan_kv_split


def _chain_tables(Z, H, Sq, lengths, signals):
    offsets, sizes, cums, lo, total = [], [], [], 0, 0
    for n in lengths:
        offsets.append([0, 0, 0, lo])
        sizes.append([Z, H, Sq, n])
        lo += n
        total += Z * H * Sq
        cums.append(total)
    return offsets, sizes, cums, signals, lo


def test_plans():
    def plan(Z, H, Sq, lengths, signals, always=False, **kw):
        offsets, sizes, cums, sigs, _ = _chain_tables(Z, H, Sq, lengths, signals)
        args = dict(causal=False, producer=False, units=256, always=always)
        args.update(kw)
        return plan_kv_split(offsets, sizes, cums, sigs, **args)

    # 48 pairs of 48 blocks, every wave behind a flag: 32 units stay free for the copies
    got = plan(2, 4, 1536, [1536] * 4, [0] * 4)
    assert got.chain and got.pairs == 48 and got.parts == 4 and got.programs <= 224
    # nothing to wait for: no unit kept back
    assert plan(2, 4, 1536, [6144] * 4, [-1] * 4).programs > 224 >= plan(2, 4, 1536, [6144] * 4, [0] * 4).programs
    # only the first wave's programs do not wait; they hold units as long as they run
    free_first = plan(1, 8, 1024, [1024] * 8, [-1] + list(range(7)))
    assert free_first.programs <= 224 and free_first.pairs == 32
    # what would be single tiles is cut only if it ends as early behind the last flag, too: parts shorter than a chunk
    assert plan(1, 8, 1024, [1024] * 8, [-1] + list(range(7)), always=True) is None
    assert plan(1, 2, 1024, [2048] * 8, [-1] + list(range(7)), always=True) is None
    assert plan(1, 2, 512, [4096] * 8, [-1] + list(range(7)), always=True).parts == 16
    assert plan(1, 8, 1024, [1024] * 8, [-1] * 8, always=True).parts == 8
    # enough pairs: stay whole where they would be chained, one part where they would be single tiles - but not where
    # they wait, on every compute unit and with all its registers, for flags that a kernel may have to raise
    assert plan(1, 32, 4096, [4096] * 8, [-1] + list(range(7))) is None
    assert plan(1, 32, 4096, [4096] * 8, [-1] * 8, always=True).parts == 1
    assert plan(1, 32, 4096, [4096] * 8, [-1] + list(range(7)), always=True) is None
    for heads in range(1, 66):
        for signals in ([-1] + list(range(7)), [-1] * 7 + [0], list(range(8))):
            for sq in (256, 1024, 3072):
                got = plan(1, heads, sq, [1024] * 8, signals, always=True)
                assert got is None or got.programs <= 224
    # tiles that need little more than a round, and whole pairs that gain as little (560 of 22 blocks: 259 us, as tiles 225)
    assert plan(1, 70, 2048, [1408] * 2, [-1, -1], always=True) is None
    assert plan(1, 40, 512, [4352] * 4, [-1, 0, 1, 2], always=True) is None
    visits = ([[0, 0, i * 1024, 0] for i in range(2)], [[1, 38, 1024, 2816]] * 2, [38 * 1024 * (i + 1) for i in range(2)], [0, 1])
    assert plan_kv_split(*visits, causal=False, producer=True, units=256, always=True) is None
    # a producer's programs end in as many rounds where a few units are taken by the kernels that wait for its flags
    for heads in range(1, 40):
        for kv in (1024, 4096, 8192):
            visits = ([[0, 0, i * 512, 0] for i in range(4)], [[1, heads, 512, kv]] * 4, [heads * 512 * (i + 1) for i in range(4)])
            got = plan_kv_split(*visits, list(range(4)), causal=False, producer=True, units=256, always=True)
            assert got is None or -(-got.programs // 256) == -(-got.programs // 240)
    # odd q blocks, unequal q ranges, a causal consumer, a q block visited twice by a producer: not cut
    assert plan(1, 2, 384, [512] * 2, [-1, 0]) is None
    assert plan(1, 2, 512, [512] * 2, [-1, 0], causal=True) is None
    assert plan(1, 2, 512, [512] * 2, [0, 1], producer=True) is None
    assert plan_kv_split([[0, 0, 0, 0], [0, 0, 256, 0]], [[1, 2, 256, 512]] * 2, [512, 1024], [-1, 0], causal=False,
                         producer=False, units=256, always=True) is None
    # a table that the checks will refuse does not stop the planner
    assert plan(1, 2, 0, [512], [-1]) is None


def _inputs(Z, H, Sq, Skv, dtype, layout="bhsd", seed=3):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(Z, H, s, 128, generator=g).to(dtype) for s in (Sq, Skv, Skv))
    return q, k, v, (lambda t: t if layout == "bhsd" else t.permute(0, 2, 1, 3).contiguous())


def _rel(out, ref):
    return ((out.float().cpu() - ref).abs().max() / ref.abs().max()).item()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Z,H,Sq,lengths,parts", [
    (1, 1, 256, [128], 1),                           # one pair, one block: nothing to cut
    (1, 1, 256, [128, 128], 2),                      # a block each
    (1, 2, 256, [128, 384, 256], 4),                 # unequal waves, parts that begin inside them
    (2, 3, 512, [128] * 7, 7),                       # three steps of the tree, an odd number of parts
    (1, 1, 512, [128 * 23, 128 * 2, 128 * 31], 16),  # the most parts
    (1, 20, 1024, [256] * 3, 5),                     # several parts, none as long as a wave
    (1, 66, 1024, [128] * 3, 1),                     # more pairs than compute units, whole
    (1, 66, 1024, [128] * 3, 3),                     # and more programs than run at a time
])
def test_parts_add_up(hip, monkeypatch, Z, H, Sq, lengths, parts, dtype):
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward

    offsets, sizes, cums, signals, Skv = _chain_tables(Z, H, Sq, lengths, [-1] + list(range(len(lengths) - 1)))
    q, k, v, _ = _inputs(Z, H, Sq, Skv, dtype)
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    kw = dict(wave_offsets=table(offsets), wave_sizes=table(sizes), cum_wave_sizes=table(cums), signal_offsets=table(signals),
              signal_ptr=torch.ones(max(len(lengths) - 1, 1), dtype=torch.int64, device="cuda"), cum_tiles=cums[-1],
              return_lse=True)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    split = KvSplit(True, Z * H * Sq // 256, parts, -(-sum(lengths) // (BLOCK * parts)))
    monkeypatch.setattr("syncopate_amd.computation.attn.template.plan_kv_split", lambda *args, **kwargs: split)
    o, lse = attention_forward(qd, kd, vd, 128 ** -0.5, **kw)
    again, lse2 = attention_forward(qd, kd, vd, 128 ** -0.5, **kw)
    check_status()
    assert torch.equal(o, again) and torch.equal(lse, lse2)          # whichever part arrives last
    # one rounding of the result and one of the probabilities (2^-9 each in bf16, 2^-12 in fp16), relative to the
    # largest value of the result; three times that
    assert _rel(o, numerics.sdpa_fp32(q, k, v, 128 ** -0.5)) <= (1.2e-2 if dtype == torch.bfloat16 else 1.5e-3)
    s = (q.float() @ k.float().transpose(-1, -2)) * 128 ** -0.5
    assert (lse.cpu() - torch.logsumexp(s, dim=-1) / 0.6931471805599453).abs().max().item() <= 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("parts,layout", [(1, "bhsd"), (2, "bshd"), (3, "bhsd"), (8, "bhsd")])
@pytest.mark.parametrize("Z,H,rows,chunks,skv", [(1, 2, 256, 4, 1024), (2, 1, 512, 3, 1536), (1, 8, 512, 8, 4096), (1, 1, 256, 1, 256)])
def test_producer_parts(hip, monkeypatch, Z, H, rows, chunks, skv, parts, layout, causal):
    """Every wave's counter reaches its tiles and every flag goes up, with the result in place."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward

    Sq = rows * chunks
    Skv = Sq if causal else skv + 128
    q, k, v, lay = _inputs(Z, H, Sq, Skv, torch.bfloat16, layout)
    split = KvSplit(False, Z * H * Sq // 256, parts, max(Skv // (BLOCK * parts), 1))
    monkeypatch.setattr("syncopate_amd.computation.attn.template.plan_kv_split", lambda *args, **kwargs: split)
    order = [(i + 1) % chunks for i in range(chunks)]
    cums = [(i + 1) * Z * H * rows for i in range(chunks)]
    flags = torch.zeros(chunks, dtype=torch.int64, device="cuda")
    counters = torch.zeros(chunks, dtype=torch.int32, device="cuda")
    o = attention_forward(lay(q).cuda(), lay(k).cuda(), lay(v).cuda(), 128 ** -0.5, wave_offsets=[[0, 0, c * rows, 0] for c in order],
                          wave_sizes=[[Z, H, rows, Skv]] * chunks, cum_wave_sizes=cums, signal_ptr=flags,
                          signal_offsets=list(range(chunks)), counter_ptr=counters, cum_tiles=cums[-1], causal=causal, layout=layout)
    check_status()
    assert counters.tolist() == [Z * H * rows // BLOCK] * chunks and flags.tolist() == [1] * chunks
    got = o if layout == "bhsd" else o.permute(0, 2, 1, 3)
    assert _rel(got, numerics.sdpa_fp32(q, k, v, 128 ** -0.5, causal=causal)) <= 1.2e-2


@pytest.mark.gpu
def test_part_of_minus_infinity(hip, monkeypatch):
    """A part in which a row's scores are all minus infinity adds nothing, as the same blocks do behind others."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward

    offsets, sizes, cums, signals, Skv = _chain_tables(1, 1, 256, [512, 512], [-1, -1])
    q, k, v, _ = _inputs(1, 1, 256, Skv, torch.bfloat16)
    monkeypatch.setattr("syncopate_amd.computation.attn.template.plan_kv_split", lambda *args, **kwargs: KvSplit(True, 1, 4, 2))
    q[..., 0] = 1.0
    k[:, :, 512:, 0] = -float("inf")
    o = attention_forward(q.cuda(), k.cuda(), v.cuda(), 128 ** -0.5, wave_offsets=offsets, wave_sizes=sizes, cum_wave_sizes=cums,
                          signal_ptr=torch.ones(1, dtype=torch.int64, device="cuda"), signal_offsets=signals, cum_tiles=cums[-1])
    check_status()
    assert _rel(o, numerics.sdpa_fp32(q, k[:, :, :512], v[:, :, :512], 128 ** -0.5)) <= 1.2e-2


@pytest.mark.gpu
def test_template_tables_are_kept_and_follow_their_source(hip):
    """The hand-written template's call keeps its converted tables: again on another stream, and after the caller has
    changed its tables in place, by whatever means; tables on the host, and a call that keeps no versions."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention, build_waves_and_signals_divisible

    q, k, v, _ = _inputs(1, 2, 512, 1024, torch.bfloat16)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    waves = build_waves_and_signals_divisible(1, 2, 512, 1024, w=4)
    want = numerics.sdpa_fp32(q, k, v, 0.1)
    side = torch.cuda.Stream()
    for stream in (None, None, side):
        torch.cuda.synchronize()
        o = attention(qd, kd, vd, 0.1, waves, stream=stream)
        torch.cuda.synchronize()
        check_status()
        assert _rel(o, want) <= 1.2e-2
    other = torch.tensor([0, 2, 4, 0], dtype=torch.int32, device="cuda")          # the last wave: the first again
    twice = torch.cat([k[:, :, :768], k[:, :, :256]], dim=2), torch.cat([v[:, :, :768], v[:, :, :256]], dim=2)
    for blocks, kv in ((other, twice), (torch.tensor([0, 2, 4, 6], dtype=torch.int32, device="cuda"), (k, v)), (other, twice)):
        if blocks is other:
            waves["wave_offsets"].data.view(4, 4)[:, 3] = blocks        # a write that the tensor's version does not count
        else:
            waves["wave_offsets"].view(4, 4)[:, 3] = blocks
        o = attention(qd, kd, vd, 0.1, waves)
        check_status()
        assert _rel(o, numerics.sdpa_fp32(q, *kv, 0.1)) <= 1.2e-2
    on_host = {n: t.tolist() if n in ("wave_offsets", "wave_sizes", "cum_wave_sizes", "signal_offsets") else t for n, t in waves.items()}
    on_host["wave_offsets"] = [on_host["wave_offsets"][i:i + 4] for i in range(0, 16, 4)]
    with torch.inference_mode():
        o = attention(qd, kd, vd, 0.1, on_host)
    check_status()
    assert _rel(o, numerics.sdpa_fp32(q, *twice, 0.1)) <= 1.2e-2


@pytest.mark.gpu
def test_template_call_is_not_captured(hip):
    """Its tables are read on every call, so that a captured launch would go on with what they held (and where they lay)."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention, build_waves_and_signals_divisible

    q, k, v, _ = _inputs(1, 2, 512, 1024, torch.bfloat16)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    waves = build_waves_and_signals_divisible(1, 2, 512, 1024, w=4)
    attention(qd, kd, vd, 0.1, waves)
    check_status()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="cannot be captured"):
            attention(qd, kd, vd, 0.1, waves)
        qd.add_(0)                                  # (an empty graph is warned about)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["explicit", "auto", "causal auto", "producer"])
def test_same_tables_with_another_number_of_waves(hip, form):
    """What the launcher worked out for the first NUM_WAVES rows of a set of tables is not taken for another number of
    rows: eight waves that share their q rows, then the same table objects with eight more over other rows."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward

    H, half, chunk, causal = 8, 1024, 256 if form == "causal auto" else 1024, form == "causal auto"
    Sq = 2 * half
    Skv = Sq if causal else 8 * chunk
    if form == "producer":
        offsets = [[0, 0, i * 128 * 2, 0] for i in range(8)]
        sizes = [[1, H, 256, Skv]] * 8
        steps, signals = (4, 8, 4), list(range(8))
    else:
        offsets = [[0, 0, rows, i * chunk] for rows in (0, half) for i in range(8)]
        sizes = [[1, H, half, chunk]] * 16
        steps, signals = (8, 16, 8), [-1] * 16
    cums = [sum(s[0] * s[1] * s[2] for s in sizes[:i + 1]) for i in range(len(sizes))]
    q, k, v, _ = _inputs(1, H, Sq, Skv, torch.bfloat16)
    want = numerics.sdpa_fp32(q, k, v, 0.1, causal=causal)
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    tables = dict(wave_offsets=table(offsets), wave_sizes=table(sizes), cum_wave_sizes=table(cums), signal_offsets=table(signals))
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    for waves in steps:
        out = torch.full_like(qd, float("nan"))
        kw = dict(form="auto") if "auto" in form else {}
        if form == "producer":
            kw = dict(counter_ptr=torch.zeros(8, dtype=torch.int32, device="cuda"))
        attention_forward(qd, kd, vd, 0.1, NUM_WAVES=waves, cum_tiles=cums[waves - 1], out=out, causal=causal,
                          signal_ptr=torch.zeros(8, dtype=torch.int64, device="cuda"), **kw, **tables)
        check_status()
        rows = max(o[2] + s[2] for o, s in zip(offsets[:waves], sizes))
        # one rounding of the result and of the probabilities, three times that; see test_parts_add_up
        assert _rel(out[:, :, :rows], want[:, :, :rows]) <= 1.2e-2
        assert bool(out[:, :, rows:].isnan().all())


@pytest.mark.gpu
@pytest.mark.parametrize("H,Sq,chunk,form,cut", [
    (2, 512, 4096, "explicit", True),
    (8, 1024, 1024, "auto", True),
    (2, 512, 2048, "auto", True),
    (20, 1024, 1024, "explicit", False),         # more tiles than run at a time, all but the first wave's waiting
    (24, 3072, 512, "explicit", False),
])
def test_flags_that_kernels_raise_while_parts_wait(hip, monkeypatch, H, Sq, chunk, form, cut):
    """The chunks' flags go up one after the other, in another order than the waves', raised by kernels that are launched
    behind the attention kernel: whatever form runs, its waiting programs leave room for them."""
    from syncopate_amd import _lib
    from syncopate_amd.communication.comm_runtime.streams import pick_side_streams
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward, template

    chunks = 8
    plans, planner = [], plan_kv_split
    monkeypatch.setattr(template, "plan_kv_split", lambda *a, **kw: plans.append(planner(*a, **kw)) or plans[-1])
    offsets, sizes, cums, signals, Skv = _chain_tables(1, H, Sq, [chunk] * chunks, [-1] + list(range(chunks - 1)))
    q, k, v, _ = _inputs(1, H, Sq, Skv, torch.bfloat16)
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    tables = dict(wave_offsets=table(offsets), wave_sizes=table(sizes), cum_wave_sizes=table(cums), signal_offsets=table(signals),
                  cum_tiles=cums[-1])
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    lib, side = _lib.load(), pick_side_streams(1)[0]
    flags = torch.ones(chunks, dtype=torch.int64, device="cuda")
    resident = attention_forward(qd, kd, vd, 128 ** -0.5, signal_ptr=flags, form=form, **tables)
    assert len(plans) == 1 and (plans[0] is not None) == cut
    for first in (0, 3):
        flags.zero_()
        torch.cuda.synchronize()
        o = attention_forward(qd, kd, vd, 128 ** -0.5, signal_ptr=flags, form=form, **tables)
        for i in range(chunks - 1):
            _lib.check("syn_delay_us", lib.syn_delay_us(30, _lib.stream_handle(side)))
            _lib.check("syn_flag_set", lib.syn_flag_set(flags.data_ptr() + 8 * ((first + 2 * i) % 7), 1, _lib.stream_handle(side)))
        check_status()
        if cut:                                  # (the other form merges in the order in which visits end)
            assert torch.equal(o, resident)
        # one rounding of the result and of the probabilities, three times that, and one of the result per merge
        assert _rel(o[:, :2], numerics.sdpa_fp32(q[:, :2], k[:, :2], v[:, :2], 128 ** -0.5)) <= (1.2e-2 if cut else 2e-2)


@pytest.mark.gpu
def test_producer_of_several_rounds_announces_its_waves_in_order(hip, monkeypatch):
    """More programs than compute units: the flags of the table's first waves go up rounds before the last one's."""
    import time

    from syncopate_amd.communication.comm_runtime.streams import pick_side_streams
    from syncopate_amd.computation._launch import check_status, compute_units
    from syncopate_amd.computation.attn import attention_forward

    H, Sq, Skv, chunks = 12, 8192, 8192, 8
    rows = Sq // chunks
    offsets, sizes = [[0, 0, i * rows, 0] for i in range(chunks)], [[1, H, rows, Skv]] * chunks
    cums = [(i + 1) * H * rows for i in range(chunks)]
    plan = KvSplit(False, 384, 2, 32)
    assert plan.programs > 2 * 256 >= 2 * compute_units(0)
    monkeypatch.setattr("syncopate_amd.computation.attn.template.plan_kv_split", lambda *args, **kwargs: plan)
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(1, H, s, 128, device="cuda", generator=g).bfloat16() for s in (Sq, Skv, Skv))
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    tables = dict(wave_offsets=table(offsets), wave_sizes=table(sizes), cum_wave_sizes=table(cums),
                  signal_offsets=table(list(range(chunks))), cum_tiles=cums[-1])
    flags = torch.zeros(chunks, dtype=torch.int64, device="cuda")
    counters = torch.zeros(chunks, dtype=torch.int32, device="cuda")
    side, seen = pick_side_streams(1)[0], torch.zeros(chunks, dtype=torch.int64).pin_memory()
    shares = []
    for _ in range(5):
        flags.zero_()
        counters.zero_()
        torch.cuda.synchronize()
        start, when = time.perf_counter(), {}
        attention_forward(q, k, v, 128 ** -0.5, signal_ptr=flags, counter_ptr=counters, **tables)
        while len(when) < chunks and time.perf_counter() - start < 10:
            with torch.cuda.stream(side):
                seen.copy_(flags, non_blocking=True)
            side.synchronize()
            for i in range(chunks):
                if int(seen[i]):
                    when.setdefault(i, time.perf_counter() - start)
        check_status()
        assert counters.tolist() == [H * rows // BLOCK] * chunks
        shares.append(when[0] / when[chunks - 1])
    # 48 of 384 pairs of the first wave end with the first of three rounds; all at the end if a wave is one XCD's
    assert sorted(shares)[2] < 0.7, shares


@pytest.mark.gpu
def test_part_that_begins_in_a_wave_of_other_rows(hip, monkeypatch):
    """The kernel compares the wave in which a part begins with the first one, whose q blocks it takes, and says so."""
    from syncopate_amd import _lib
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward, template

    q, k, v, _ = _inputs(1, 1, 512, 512, torch.bfloat16)
    monkeypatch.setattr(template, "plan_kv_split", lambda *args, **kwargs: KvSplit(True, 1, 2, 2))
    monkeypatch.setattr(template, "already_checked", lambda *args: True)
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    attention_forward(q.cuda(), k.cuda(), v.cuda(), 0.1, wave_offsets=table([[0, 0, 0, 0], [0, 0, 256, 256]]),
                      wave_sizes=table([[1, 1, 256, 256]] * 2), cum_wave_sizes=table([256, 512]), signal_offsets=table([-1, -1]),
                      signal_ptr=torch.ones(1, dtype=torch.int64, device="cuda"), cum_tiles=512)
    with pytest.raises(RuntimeError, match=rf"kernel status \[{_lib.SYN_STATUS_BAD_CHAIN}, 1, "):
        check_status()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["split", "auto split", "auto chain", "auto list", "causal auto", "producer"])
def test_new_tables_are_read_back_once(hip, monkeypatch, kind):
    """Tables that the launcher has not seen cost one read-back, whatever it works out from them; tables it has seen and
    tables on the host cost none."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward, template

    rows = 512 if kind in ("auto list", "producer") else 256
    offsets = [[0, 0, i * 256 if rows == 512 else 0, 256 * i] for i in range(2)]
    sizes, cums, signals = [[1, 2, 256, 256]] * 2, [512, 1024], [0, 1]
    causal = kind == "causal auto"
    q, k, v, _ = _inputs(1, 2, 512 if causal else rows, 512, torch.bfloat16)
    q, k, v = q.cuda(), k.cuda(), v.cuda()
    read, copies = [], template.host_copies
    monkeypatch.setattr(template, "host_copies", lambda tables: read.append(len(tables)) or copies(tables))
    monkeypatch.setattr(template, "host_copy", lambda table: pytest.fail("read back by itself"))
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    kw = dict(form="auto" if "auto" in kind else "explicit", causal=causal, signal_ptr=torch.ones(2, dtype=torch.int64, device="cuda"))
    if "split" in kind:
        monkeypatch.setattr(template, "plan_kv_split", lambda *args, **kwargs: KvSplit(True, 2, 2, 2))
    for given, count in ((table, 1), (lambda x: x, 0)):
        tables = dict(wave_offsets=given(offsets), wave_sizes=given(sizes), cum_wave_sizes=given(cums), signal_offsets=given(signals))
        read.clear()
        for _ in range(2):
            if kind == "producer":
                kw["counter_ptr"] = torch.zeros(2, dtype=torch.int32, device="cuda")
            attention_forward(q, k, v, 0.1, cum_tiles=1024, **kw, **tables)
        assert read == [4] * count
    check_status()


@pytest.mark.gpu
@pytest.mark.parametrize("producer", [False, True])
def test_captured_split(hip, producer):
    """A planned split under graph capture: every replay starts from zeroed words of its own, with eager launches of the
    same tables between the replays."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward

    H, chunks, scale = 8, 8, 128 ** -0.5
    Sq, Skv = (2048, 4096) if producer else (1024, 8192)
    rows = Sq // chunks
    if producer:
        offsets, sizes = [[0, 0, i * rows, 0] for i in range(chunks)], [[1, H, rows, Skv]] * chunks
        cums = [(i + 1) * H * rows for i in range(chunks)]
    else:
        offsets, sizes, cums, _, _ = _chain_tables(1, H, Sq, [Skv // chunks] * chunks, None)
    signals = list(range(chunks)) if producer else [-1] * chunks
    plan = plan_kv_split(offsets, sizes, cums, signals, causal=False, producer=producer, units=256, always=True)
    assert plan.parts > 1 and plan.chain != producer
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    tables = dict(wave_offsets=table(offsets), wave_sizes=table(sizes), cum_wave_sizes=table(cums), signal_offsets=table(signals),
                  cum_tiles=cums[-1])
    flags = torch.full((chunks,), 0 if producer else 1, dtype=torch.int64, device="cuda")
    counters = torch.zeros(chunks, dtype=torch.int32, device="cuda") if producer else None
    q, k, v = (t.cuda() for t in _inputs(1, H, Sq, Skv, torch.bfloat16)[:3])
    out = torch.zeros_like(q)

    def launch(into):
        if producer:
            flags.zero_()
            counters.zero_()
        return attention_forward(q, k, v, scale, signal_ptr=flags, counter_ptr=counters, out=into, **tables)

    launch(out)                                          # warm-up: tables planned and checked
    check_status()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph):
            launch(out)
    torch.cuda.current_stream().wait_stream(side)
    for replay in range(4):
        nq, nk, nv, _ = _inputs(1, H, Sq, Skv, torch.bfloat16, seed=40 + replay)
        q.copy_(nq.cuda()); k.copy_(nk.cuda()); v.copy_(nv.cuda())
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        for _ in range(2):                               # again at once: behind the first one's words
            graph.replay()
        torch.cuda.synchronize()
        check_status()
        assert flags.tolist() == [1] * chunks
        assert _rel(out, numerics.sdpa_fp32(nq, nk, nv, scale)) <= 1.2e-2, f"replay {replay}"
        assert torch.equal(out, launch(torch.empty_like(q))), f"replay {replay}"
        check_status()


@pytest.mark.gpu
def test_producer_beside_a_kernel_that_waits_for_its_flags(hip):
    """An exchange waits for a producer's flags by kernels on side streams; they cost the producer no round of programs."""
    from syncopate_amd import _lib
    from syncopate_amd.communication.comm_runtime.streams import pick_side_streams
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward

    lib, side, H, Sq, Skv, chunks = _lib.load(), pick_side_streams(1)[0], 8, 2048, 8192, 8
    rows = Sq // chunks
    offsets, sizes = [[0, 0, i * rows, 0] for i in range(chunks)], [[1, H, rows, Skv]] * chunks
    cums = [(i + 1) * H * rows for i in range(chunks)]
    assert plan_kv_split(offsets, sizes, cums, list(range(chunks)), causal=False, producer=True, units=256, always=True)
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(1, H, s, 128, device="cuda", generator=g).bfloat16() for s in (Sq, Skv, Skv))
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    tables = dict(wave_offsets=table(offsets), wave_sizes=table(sizes), cum_wave_sizes=table(cums),
                  signal_offsets=table(list(range(chunks))), cum_tiles=cums[-1])
    flags = torch.zeros(chunks, dtype=torch.int64, device="cuda")
    counters = torch.zeros(chunks, dtype=torch.int32, device="cuda")
    times = {0: [], 1: []}
    for waiting in (0, 1) * 6:
        flags.zero_()
        counters.zero_()
        torch.cuda.synchronize()
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        if waiting:
            _lib.check("syn_flag_wait", lib.syn_flag_wait(flags.data_ptr() + 8 * (chunks - 1), 1, 2_000_000, None,
                                                          _lib.stream_handle(side)))
        torch.cuda._sleep(1_000_000)             # the launch is queued before the clock starts
        start.record()
        attention_forward(q, k, v, 128 ** -0.5, signal_ptr=flags, counter_ptr=counters, **tables)
        end.record()
        check_status()
        times[waiting].append(start.elapsed_time(end))
    assert min(times[1]) <= 1.25 * min(times[0]), times          # a round more is 1.5
