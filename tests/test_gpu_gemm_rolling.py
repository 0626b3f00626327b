"""Programs of the GEMM that go on from one tile's K loop into the next one's: the same bits as one program per tile, for numbers
of slabs around the pipelines' depth, with flags that are up, that come late, and that come out of order."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _table(rows):
    return torch.tensor(rows, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("bm,bn", [(128, 128), (128, 256), (256, 128), (256, 256), (256, 224)])
@pytest.mark.parametrize("slabs", [1, 2, 3, 4, 5, 6, 7, 12])
def test_same_bits_as_a_program_per_tile(hip, slabs, bm, bn):
    from syncopate_amd.computation._launch import check_status, trust_flags
    from syncopate_amd.computation.gemm import gemm_consumer, gemm_producer

    world, k = 3, 64 * slabs
    rows, n = 2 * bm, 3 * bn
    m = world * rows
    g = torch.Generator(device="cuda").manual_seed(slabs)
    a, b = ((0.1 * torch.randn(s, k, device="cuda", generator=g)).bfloat16() for s in (m, n))
    want = a.float() @ b.float().T
    sizes, offsets, signals = _table([[rows, n]] * world), _table([[i * rows, 0] for i in (1, 2, 0)]), _table([-1, 1, 0])
    flags = torch.ones(2, dtype=torch.int64, device="cuda")
    trust_flags(flags)
    log = torch.empty(m // bm * (n // bn), 4, dtype=torch.int32, device="cuda")      # (and no smaller kernel tile)
    results = []
    for programs in (256, 5, 2, 1):            # 18 tiles
        c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        gemm_consumer(a, b, c, flags, sizes, offsets, signals, world, programs, bm, bn, 64, 2, cum_tiles=m * n, visit_log=log)
        results.append(c)
        c = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        done = torch.zeros(world, dtype=torch.int64, device="cuda")
        counts = torch.zeros(world, dtype=torch.int32, device="cuda")
        gemm_producer(a, b, c, done, sizes, offsets, _table([2, 0, 1]), programs, bm, bn, 64, 2, cum_tiles=m * n, visit_log=log,
                      counter_buffer=counts)
        assert done.tolist() == [1] * world and counts.tolist() == [6] * world
        results.append(c)
    check_status()
    # one rounding of the result (2^-9 of a value), sums of up to 768 products in 32 bits; twice that
    assert (results[0].float() - want).abs().max() <= 4e-3 * want.abs().max()
    assert all(torch.equal(c, results[0]) for c in results)


@pytest.mark.parametrize("trusted", [True, False])
@pytest.mark.parametrize("waves,order", [(6, [0, 1, 2, 3, 4]), (6, [4, 2, 3, 0, 1]), (70, None)])
def test_flags_that_come_late(hip, trusted, waves, order):
    """Flags raised one after the other by kernels behind the GEMM; more waves than are looked at at a time."""
    from syncopate_amd import _lib
    from syncopate_amd.communication.comm_runtime.streams import pick_side_streams
    from syncopate_amd.computation._launch import check_status, trust_flags
    from syncopate_amd.computation.gemm import gemm_consumer

    rows, n, k, bm, bn = 128, 512, 256, 128, 128
    m = waves * rows
    g = torch.Generator(device="cuda").manual_seed(waves)
    a, b = ((0.1 * torch.randn(s, k, device="cuda", generator=g)).half() for s in (m, n))
    sizes, offsets, signals = _table([[rows, n]] * waves), _table([[i * rows, 0] for i in range(waves)]), _table(list(range(-1, waves - 1)))
    flags = torch.ones(waves, dtype=torch.int64, device="cuda")
    if trusted:
        trust_flags(flags)
    lib, side = _lib.load(), pick_side_streams(1)[0]

    def run():
        c = torch.full((m, n), float("nan"), dtype=torch.half, device="cuda")
        gemm_consumer(a, b, c, flags, sizes, offsets, signals, waves, 7, bm, bn, 64, 8, cum_tiles=m * n)
        return c

    resident = run()
    assert (resident.float() - a.float() @ b.float().T).abs().max() <= 4e-3 * resident.float().abs().max()
    flags.zero_()
    torch.cuda.synchronize()
    late = run()
    for i in order or range(waves - 1):
        _lib.check("syn_delay_us", lib.syn_delay_us(10, _lib.stream_handle(side)))
        _lib.check("syn_flag_set", lib.syn_flag_set(flags.data_ptr() + 8 * i, 1, _lib.stream_handle(side)))
    check_status()
    assert torch.equal(late, resident)
