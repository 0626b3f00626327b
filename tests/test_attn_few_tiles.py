"""form="auto" on all-to-all tables: the visits are planned where there are more tiles with work than compute units, and run as
single tiles where there are not."""

import pytest
import torch

from oracle import numerics

pytestmark = pytest.mark.gpu


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
