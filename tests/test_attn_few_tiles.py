"""form="auto" on all-to-all tables: the visits are planned where there are more tiles with work than compute units, and run as
single tiles where there are not, unless a plan keeps sums of several visits in 32 bits."""

import random

import pytest
import torch

from oracle import numerics
from syncopate_amd.computation.attn.work_plan import WORK_CONTINUES, chains_visits, plan_attention_work, table_visits


def _tables(H, chunks):
    """The all-to-all table of chunks of these rows."""
    starts, offsets, sizes, signals, cums = [sum(chunks[:i]) for i in range(len(chunks))], [], [], [], []
    for w in range(len(chunks)):
        for q, kv in [(w, w)] + [pair for p in range(w) for pair in ((p, w), (w, p))]:
            offsets.append([0, 0, starts[q], starts[kv]])
            sizes.append([1, H, chunks[q], chunks[kv]])
            signals.append(w - 1)
            cums.append((cums[-1] if cums else 0) + H * chunks[q])
    return offsets, sizes, cums, signals


def test_chained_visits_are_foreseen():
    rng, seen = random.Random(4), set()
    for _ in range(400):
        H, units = rng.choice([1, 2, 3, 8]), rng.choice([16, 64, 256])
        tables = _tables(H, [256 * rng.choice([1, 1, 1, 2, 4, 16]) for _ in range(rng.randint(1, 6))])[:3]
        for causal in (False, True):
            plan = plan_attention_work(*tables, causal=causal, num_programs=units, max_blocks="fair")
            chained = any(word & WORK_CONTINUES for entries in plan.program_entries for word in entries)
            assert chains_visits(table_visits(*tables, causal=causal), units) == chained
            seen.add(chained)
    assert seen == {False, True}


@pytest.mark.gpu
@pytest.mark.parametrize("H,chunks,causal", [(1, (256, 4096, 1024, 256, 256), False), (2, (256, 256, 4096), False),
                                             (3, (4096, 1024, 256, 256, 256), True)])
def test_chained_visits_stay_planned(hip, monkeypatch, H, chunks, causal):
    """Fewer tiles than units, but visits of uneven chunks that a plan chains: planned, so that no sum of theirs is rounded to 16 bits."""
    from syncopate_amd.computation._launch import check_status, compute_units
    from syncopate_amd.computation.attn import attention_forward, template

    offsets, sizes, cums, signals = _tables(H, chunks)
    tiles = sum(not causal or o[2] + q >= o[3] + 128 for o, s in zip(offsets, sizes) for q in range(128, s[2] + 1, 128)) * H
    assert tiles <= compute_units(0)
    planned, planner = [], template.plan_attention_work
    monkeypatch.setattr(template, "plan_attention_work", lambda *args, **kw: planned.append(planner(*args, **kw)) or planned[-1])
    g = torch.Generator().manual_seed(H)
    q, k, v = (torch.randn(1, H, sum(chunks), 128, generator=g).bfloat16() for _ in range(3))
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    o = attention_forward(q.cuda(), k.cuda(), v.cuda(), 128 ** -0.5, wave_offsets=table(offsets), wave_sizes=table(sizes),
                          cum_wave_sizes=table(cums), signal_offsets=table(signals), cum_tiles=cums[-1], causal=causal, form="auto",
                          signal_ptr=torch.ones(len(chunks), dtype=torch.int64, device="cuda"))
    check_status()
    assert len(planned) == 1 and any(word & WORK_CONTINUES for entries in planned[0].program_entries for word in entries)
    want = numerics.sdpa_fp32(q, k, v, 128 ** -0.5, causal=causal)
    # roundings of the result, of the probabilities and of up to five merges, 2^-9 each of the largest value
    assert (o.float().cpu() - want).abs().max() <= 2e-2 * want.abs().max()


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("H,chunk,chunks", [(2, 256, 2), (8, 512, 2), (16, 512, 2), (17, 512, 2), (21, 512, 2), (22, 512, 2), (2, 256, 8)])
def test_planned_only_for_more_tiles_than_units(hip, monkeypatch, H, chunk, chunks, causal):
    from syncopate_amd.computation._launch import check_status, compute_units
    from syncopate_amd.computation.attn import attention_forward, template

    offsets, sizes, signals = [], [], []
    for w in range(chunks):
        for q, kv in [(w, w)] + [pair for p in range(w) for pair in ((p, w), (w, p))]:
            offsets.append([0, 0, q * chunk, kv * chunk])
            sizes.append([1, H, chunk, chunk])
            signals.append(w - 1)
    cums = [(i + 1) * H * chunk for i in range(len(sizes))]
    # under a causal mask the visits of an earlier chunk to a later one have no work
    tiles = H * chunk // 128 * sum(not causal or o[2] >= o[3] for o in offsets)
    planned, planner = [], template.plan_attention_work
    monkeypatch.setattr(template, "plan_attention_work", lambda *args, **kw: planned.append(1) or planner(*args, **kw))
    g = torch.Generator().manual_seed(H)
    q, k, v = (torch.randn(1, H, chunk * chunks, 128, generator=g).bfloat16() for _ in range(3))
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    tables = dict(wave_offsets=table(offsets), wave_sizes=table(sizes), cum_wave_sizes=table(cums), signal_offsets=table(signals),
                  cum_tiles=cums[-1])
    flags = torch.ones(chunks, dtype=torch.int64, device="cuda")
    for _ in range(2):
        o = attention_forward(q.cuda(), k.cuda(), v.cuda(), 128 ** -0.5, signal_ptr=flags, causal=causal, form="auto", **tables)
        check_status()
        want = numerics.sdpa_fp32(q[:, :2], k[:, :2], v[:, :2], 128 ** -0.5, causal=causal)
        # roundings of the result, of the probabilities and of up to eight merges, 2^-9 each of the largest value
        assert (o[:, :2].float().cpu() - want).abs().max() <= 2e-2 * want.abs().max()
    assert len(planned) == (tiles > compute_units(0))
