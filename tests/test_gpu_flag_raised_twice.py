"""Launches on flags that nobody vouches for (SYN_GEMM_ACQUIRE_ALWAYS, SYN_ATTN_ACQUIRE_ALWAYS): a flag that is up when the kernel
begins, goes down before the kernel gets to its wave and up again behind new data is waited for."""

import pytest
import torch

from syncopate_amd import _lib
from syncopate_amd.computation._launch import check_status

pytestmark = pytest.mark.gpu


def _again(launch, flags, write_new):
    """`launch` on the current stream, whose first wave takes some milliseconds, and meanwhile the second wave's flag down, new data
    20 ms later, the flag up."""
    from syncopate_amd.communication.comm_runtime.streams import pick_side_streams

    lib, side = _lib.load(), pick_side_streams(1)[0]
    launch()
    torch.cuda.synchronize()
    out = launch()
    with torch.cuda.stream(side):
        handle = _lib.stream_handle(side)
        _lib.check("syn_delay_us", lib.syn_delay_us(200, handle))
        _lib.check("syn_flag_set", lib.syn_flag_set(flags.data_ptr() + 8, 0, handle))
        _lib.check("syn_delay_us", lib.syn_delay_us(20000, handle))
        write_new()
        _lib.check("syn_flag_set", lib.syn_flag_set(flags.data_ptr() + 8, 1, handle))
    check_status()
    torch.cuda.synchronize()
    return out.clone()


@pytest.mark.parametrize("block_n", [128, 256])
def test_gemm(hip, block_n):
    from syncopate_amd.computation.gemm import gemm_consumer

    rows, n, k = 128 * 128, block_n, 8192
    g = torch.Generator(device="cuda").manual_seed(1)
    randn = lambda *shape: (0.1 * torch.randn(shape, device="cuda", generator=g)).bfloat16()
    a, b, new = randn(rows + 128, k), randn(n, k), randn(128, k)
    c = torch.zeros(rows + 128, n, dtype=torch.bfloat16, device="cuda")
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    sizes, offsets, signals = table([[rows, n], [128, n]]), table([[0, 0], [rows, 0]]), table([0, 1])
    flags = torch.ones(2, dtype=torch.int64, device="cuda")

    def launch():                                        # one program: 128 tiles of 50 to 90 us, then the last
        gemm_consumer(a, b, c, flags, sizes, offsets, signals, 1, 1, 128, block_n, 64, 8, cum_tiles=c.numel())
        return c

    got = _again(launch, flags, lambda: a[rows:].copy_(new))
    launch()
    assert torch.equal(got, c)


@pytest.mark.parametrize("form", ["dealt", "parts", "chained", "tiles"])
def test_attention(hip, monkeypatch, form):
    from syncopate_amd.computation.attn import attention_forward, template
    from syncopate_amd.computation.attn.kv_split import KvSplit

    blocks = 2000                                        # of 2.4 or 2.8 us each, on one or two programs
    whole = KvSplit(True, 1, 1, blocks + 1)
    monkeypatch.setattr(template, "plan_kv_split", lambda *args, **kwargs: whole if form == "parts" else None)
    monkeypatch.setattr(template, "plan_kv_deal", lambda *args, **kwargs: whole if form == "dealt" else None)
    g = torch.Generator(device="cuda").manual_seed(1)
    q, k, v = (torch.randn(1, 1, s, 128, device="cuda", generator=g).bfloat16() for s in (256, 128 * (blocks + 1), 128 * (blocks + 1)))
    v[:, :, 128 * blocks:] = 0
    new = torch.full((1, 1, 128, 128), 100.0, dtype=torch.bfloat16, device="cuda")
    table = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    tables = dict(wave_offsets=table([[0, 0, 0, 0], [0, 0, 0, 128 * blocks]]), wave_sizes=table([[1, 1, 256, 128 * blocks], [1, 1, 256, 128]]),
                  cum_wave_sizes=table([256, 512]), signal_offsets=table([0, 1]), cum_tiles=512)
    flags = torch.ones(2, dtype=torch.int64, device="cuda")
    options = dict(chained=dict(pair_q_blocks=True, chain_q_blocks=True), tiles=dict(num_programs=2)).get(form, {})
    launch = lambda: attention_forward(q, k, v, 128 ** -0.5, signal_ptr=flags, **tables, **options)
    got = _again(launch, flags, lambda: v[:, :, 128 * blocks:].copy_(new))
    assert torch.equal(got, launch())
    check_status()
