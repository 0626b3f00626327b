"""Tiles behind the last full round that run as 128x128 ones: the same bits as whole, with waves that end within them."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _table(rows):
    return torch.tensor(rows, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("slabs", [10, 14, 32])
@pytest.mark.parametrize("bm,bn", [(128, 256), (256, 128), (256, 256)])
def test_same_bits_as_whole_tiles(hip, bm, bn, slabs):
    from syncopate_amd.computation._launch import check_status, trust_flags
    from syncopate_amd.computation.gemm import gemm_consumer, gemm_producer

    k, n = 64 * slabs, 3 * bn
    heights = [2, 1, 3, 1]                            # 21 tiles in waves of 6, 3, 9 and 3
    starts = [0, 2, 3, 6]
    m = 7 * bm
    g = torch.Generator(device="cuda").manual_seed(slabs)
    a, b = ((0.1 * torch.randn(s, k, device="cuda", generator=g)).bfloat16() for s in (m, n))
    sizes, offsets = _table([[h * bm, n] for h in heights]), _table([[s * bm, 0] for s in starts])
    gates, signals = _table([-1, 1, 0, 2]), _table([3, 0, -1, 1])
    flags = torch.ones(3, dtype=torch.int64, device="cuda")
    trust_flags(flags)
    log = torch.empty(21, 4, dtype=torch.int32, device="cuda")                 # (whole tiles)
    want = None
    for programs in (256, 20, 17, 16, 9, 5, 1):       # 21 tiles: 1, 4, 5, 3 and 1 of them behind full rounds, and none
        for whole in (True, False):
            c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
            gemm_consumer(a, b, c, flags, sizes, offsets, gates, 1, programs, bm, bn, 64, 2, cum_tiles=m * n, visit_log=log if whole else None)
            if want is None:
                want = c
                full = a.float() @ b.float().T
                # one rounding of the result (2^-9 of a value), sums of up to 2048 products in 32 bits; twice that
                assert (c.float() - full).abs().max() <= 4e-3 * full.abs().max()
            assert torch.equal(c, want), (programs, whole)
            c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
            done = torch.zeros(4, dtype=torch.int64, device="cuda")
            gemm_producer(a, b, c, done, sizes, offsets, signals, programs, bm, bn, 64, 2, cum_tiles=m * n, visit_log=log if whole else None)
            assert torch.equal(c, want) and done.tolist() == [1, 1, 0, 1], (programs, whole)
    check_status()


@pytest.mark.parametrize("late", [0, 3])
def test_flags_that_come_late(hip, late):
    """The flag of a wave that begins within the cut tiles, and of one that they are the only tiles of."""
    from syncopate_amd import _lib
    from syncopate_amd.communication.comm_runtime.streams import pick_side_streams
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.gemm import gemm_consumer

    bm, bn, k, n = 128, 256, 1024, 512
    m = 8 * bm                                        # 16 tiles, eight waves of two: 12 on whole tiles, 4 cut on 6 programs
    g = torch.Generator(device="cuda").manual_seed(late)
    a, b = ((0.1 * torch.randn(s, k, device="cuda", generator=g)).half() for s in (m, n))
    sizes, offsets, signals = _table([[bm, n]] * 8), _table([[i * bm, 0] for i in range(8)]), _table(list(range(8)))
    flags = torch.ones(8, dtype=torch.int64, device="cuda")
    lib, side = _lib.load(), pick_side_streams(1)[0]

    def run():
        c = torch.full((m, n), float("nan"), dtype=torch.half, device="cuda")
        gemm_consumer(a, b, c, flags, sizes, offsets, signals, 8, 6, bm, bn, 64, 2, cum_tiles=m * n)
        return c

    resident = run()
    assert (resident.float() - a.float() @ b.float().T).abs().max() <= 4e-3 * resident.float().abs().max()
    flags[late:].zero_()
    torch.cuda.synchronize()
    c = run()
    for i in range(late, 8):
        _lib.check("syn_delay_us", lib.syn_delay_us(10, _lib.stream_handle(side)))
        _lib.check("syn_flag_set", lib.syn_flag_set(flags.data_ptr() + 8 * i, 1, _lib.stream_handle(side)))
    check_status()
    assert torch.equal(c, resident)


@pytest.mark.parametrize("bm,bn", [(128, 256), (256, 256)])
def test_peers_rows_and_sums(hip, bm, bn):
    """A's rows from a peer's shard; C's tiles added into a peer's buffer."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.gemm import gemm_ag_direct_read, gemm_rs_producer_persistent

    world, k = 3, 1024
    rows, n = 2 * bm, 3 * bn
    m = world * rows
    g = torch.Generator(device="cuda").manual_seed(bm)
    a, b = ((0.1 * torch.randn(s, k, device="cuda", generator=g)).bfloat16() for s in (m, n))
    order = [1, 2, 0]
    sizes, offsets = _table([[rows, n]] * world), _table([[i * rows, 0] for i in order])
    log = torch.empty(18, 4, dtype=torch.int32, device="cuda")                 # (whole tiles)
    results = []
    for programs in (256, 16, 7, 5, 2):               # 18 tiles in waves of six: on 5 and on 2, a program's next tile may be its wave's
        for whole in (True, False):
            kw = dict(visit_log=log) if whole else {}
            c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
            gemm_ag_direct_read(list(a.view(world, rows, k)), b, c, sizes, offsets, order, world, world, programs, True, bm, bn, 64, 2, **kw)
            results.append(c)
            c = torch.zeros(m, n, dtype=torch.bfloat16, device="cuda")
            gemm_rs_producer_persistent(a, b, list(c.view(world, rows, n)), sizes, offsets, order, world, world, programs, bm, bn, 64, 2, **kw)
            results.append(c)
    check_status()
    want = a.float() @ b.float().T
    # one rounding of the result (2^-9 of a value), sums of 1024 products in 32 bits; twice that
    assert (results[0].float() - want).abs().max() <= 4e-3 * want.abs().max()
    assert all(torch.equal(c, results[0]) for c in results)
