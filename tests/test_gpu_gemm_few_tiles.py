"""GEMMs of few tiles, which run on smaller kernel tiles: the rule, and every form against the fp32 product."""

import pytest
import torch

from syncopate_amd.computation.gemm.tile_policy import SLAB_US, choose_kernel_tile


def test_rule():
    assert choose_kernel_tile(42, 256, 2752, 256, 256) == (128, 128)
    assert choose_kernel_tile(104, 256, 960, 256, 256) == (256, 128)
    assert choose_kernel_tile(256, 256, 8192, 256, 256) == (256, 256)       # a whole round
    assert choose_kernel_tile(129, 256, 8192, 128, 256) == (128, 256)       # twice as many would be two rounds
    assert choose_kernel_tile(128, 256, 512, 128, 256, waiting=1.0, room=224) == (128, 256)
    assert choose_kernel_tile(128, 256, 8192, 128, 256, waiting=0.75, room=224) == (128, 128)
    # a launch that waits gains more than its copies lose
    assert choose_kernel_tile(128, 256, 512, 128, 256) == (128, 128)
    assert choose_kernel_tile(128, 256, 512, 128, 256, waiting=0.75, room=224) == (128, 256)
    assert choose_kernel_tile(48, 256, 1024, 256, 256, waiting=0.75, room=224) == (256, 256)
    assert choose_kernel_tile(84, 256, 2752, 256, 256, waiting=0.75, room=224) == (256, 128)
    assert choose_kernel_tile(16, 256, 512, 256, 224) == (256, 224)         # no tile divides it
    assert choose_kernel_tile(16, 0, 512, 256, 256) == (256, 256)           # the library names the error
    assert choose_kernel_tile(200, 1024, 2048, 256, 256, units=256) == (256, 256)     # more programs than run at a time
    assert choose_kernel_tile(60, 1024, 2048, 256, 256, units=256) == (128, 128)
    for tiles in range(1, 257, 5):
        for shape in SLAB_US:
            bm, bn = choose_kernel_tile(tiles, 224, 1024, *shape, waiting=0.5, room=192)
            assert shape[0] % bm == 0 and shape[1] % bn == 0
            cut = tiles * (shape[0] // bm) * (shape[1] // bn)
            assert cut == tiles or (cut <= 224 and cut * 0.5 <= 192)


def _table(x):
    return torch.tensor(x, dtype=torch.int32, device="cuda")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("world,rows,n,k,bm,bn,programs", [
    (2, 256, 256, 64, 256, 256, 256),            # two tiles, one slab
    (4, 512, 768, 320, 256, 256, 224),           # 24 -> 96
    (3, 512, 2560, 192, 256, 256, 224),          # 60 -> 120: four times as many would not fit
    (2, 384, 1280, 1984, 128, 256, 256),         # odd numbers of tiles per wave
    (3, 256, 640, 2112, 256, 128, 100),
])
@pytest.mark.parametrize("form", ["consumer", "producer", "direct"])
def test_few_tiles(hip, form, world, rows, n, k, bm, bn, programs, dtype):
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.gemm import gemm_consumer, gemm_producer, gemm_rs_producer_persistent

    g = torch.Generator(device="cuda").manual_seed(k + n)
    m = world * rows
    a = (0.05 * torch.randn(m, k, device="cuda", generator=g)).to(dtype)
    b = (0.05 * torch.randn(n, k, device="cuda", generator=g)).to(dtype)
    sizes, offsets = _table([[rows, n]] * world), _table([[(i + 1) % world * rows, 0] for i in range(world)])
    if form == "direct":
        c = torch.zeros(world, rows, n, dtype=dtype, device="cuda")
        gemm_rs_producer_persistent(a, b, list(c), sizes, offsets, _table([(i + 1) % world for i in range(world)]), world, world,
                                    programs, bm, bn, 64, 8)
        c = c.view(m, n)
    else:
        c = torch.full((m, n), float("nan"), dtype=dtype, device="cuda")
        flags = torch.full((world,), 1 if form == "consumer" else 0, dtype=torch.int64, device="cuda")
        args = (a, b, c, flags, sizes, offsets, _table(list(range(world))))
        if form == "consumer":
            gemm_consumer(*args, world, programs, bm, bn, 64, 8, cum_tiles=m * n)
            # the same bits as on the tiles that were asked for, which a visit log shows
            whole = torch.empty_like(c)
            log = torch.zeros(m // bm * (n // bn), 4, dtype=torch.int32, device="cuda")
            gemm_consumer(a, b, whole, *args[3:], world, programs, bm, bn, 64, 8, cum_tiles=m * n, visit_log=log)
            assert torch.equal(c, whole)
        else:
            gemm_producer(*args, programs, bm, bn, 64, 8, cum_tiles=m * n)
            assert flags.tolist() == [1] * world
            # a caller that brings the counters finds its own tiles counted
            flags.zero_()
            counters = torch.zeros(world, dtype=torch.int32, device="cuda")
            gemm_producer(*args, programs, bm, bn, 64, 8, cum_tiles=m * n, counter_buffer=counters)
            assert counters.tolist() == [rows // bm * (n // bn)] * world and flags.tolist() == [1] * world
    check_status()
    ref = a.double() @ b.double().t()
    # one rounding of the result (2^-9, 2^-12 of a value, at most that of the largest); the sums are 32-bit
    assert ((c.double() - ref).abs().max() / ref.abs().max()).item() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)


@pytest.mark.gpu
@pytest.mark.parametrize("world,rows,n,k,bm,bn", [(4, 512, 768, 320, 256, 256), (2, 384, 1280, 1984, 128, 256), (3, 256, 640, 2112, 256, 128)])
@pytest.mark.parametrize("form", ["producer", "direct", "gathered", "split k"])
def test_same_bits_as_on_the_whole_tiles(hip, monkeypatch, form, world, rows, n, k, bm, bn):
    """The cut changes no bit of any form's result: the K phase is that of the caller's tile (each sum of an adding form
    goes to a zero; split K adds twice, and the sum of two does not depend on their order)."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.gemm import (gemm_ag_direct_read, gemm_producer, gemm_rs_producer_persistent, gemm_splitk, template,
                                                template_remote)

    g = torch.Generator(device="cuda").manual_seed(k + n)
    m = world * rows
    a = (0.05 * torch.randn(m, k, device="cuda", generator=g)).bfloat16()
    b = (0.05 * torch.randn(n, k, device="cuda", generator=g)).bfloat16()
    order = [(i + 1) % world for i in range(world)]
    sizes, offsets, ranks = _table([[rows, n]] * world), _table([[i * rows, 0] for i in order]), _table(order)
    rule, taken, results = choose_kernel_tile, [], []
    for cut in (True, False):
        choose = lambda *args, **kw: taken.append((args[3:5], rule(*args, **kw) if cut else args[3:5])) or taken[-1][1]
        monkeypatch.setattr(template, "choose_kernel_tile", choose)
        monkeypatch.setattr(template_remote, "choose_kernel_tile", choose)
        c = torch.zeros(world, rows, n, dtype=torch.bfloat16, device="cuda")
        if form == "producer":
            flags = torch.zeros(world, dtype=torch.int64, device="cuda")
            gemm_producer(a, b, c.view(m, n), flags, sizes, offsets, ranks, 256, bm, bn, 64, 8, cum_tiles=m * n)
            assert flags.tolist() == [1] * world
        elif form == "direct":
            gemm_rs_producer_persistent(a, b, list(c), sizes, offsets, ranks, world, world, 256, bm, bn, 64, 8)
        elif form == "gathered":
            gemm_ag_direct_read(list(a.view(world, rows, k)), b, c.view(m, n), sizes, offsets, ranks, world, world, 256, True, bm, bn, 64, 8)
        else:
            half = k // 128 * 64
            gemm_splitk(a, b, c.view(m, n), world, 256, bm, bn, 64, 8, cur_wave_sizes=_table([[m, n, half], [m, n, k - half]]),
                        wave_offsets=_table([[0, 0, 0], [0, 0, half]]), cum_tiles=2 * m * n)
        check_status()
        results.append(c)
    assert taken[0][0] != taken[0][1] and len(taken) == 2
    assert torch.equal(*results)
