"""The native steady-state launches (csrc/launch.cpp): taken for operands and tables that came through a launcher before, left to
the launcher's general path for everything else."""

import threading

import pytest
import torch

from syncopate_amd import _lib


def _table(rows):
    return torch.tensor(rows, dtype=torch.int32, device="cuda")


def test_everything_unusual_is_left_alone():
    native = _lib.native()
    host = torch.zeros(2, 4, 8, dtype=torch.bfloat16)
    assert native.reduce(host, host[0], host.view(8, 8), 0, 0) is None            # not in device memory
    assert native.reduce(None, 1, "x", 0, 0) is None and native.reduce() is None
    assert native.gemm(*[host[0]] * 7, *[0] * 10) is None and native.gemm(host) is None
    assert native.remote(host[0], host[0], [host[0]], *[host[0]] * 4, *[0] * 10) is None
    assert native.attention(*[host] * 3, 0.1, *[host] * 5, *[0] * 5, None, None, 0, 0) is None


def _gemm_case(form):
    from syncopate_amd.computation.gemm import gemm_consumer, gemm_producer, gemm_rs_producer_persistent, template, template_remote

    world, rows, n, k = 2, 256, 512, 192
    m = world * rows
    g = torch.Generator(device="cuda").manual_seed(3)
    a, b = ((0.1 * torch.randn(s, k, device="cuda", generator=g)).bfloat16() for s in (m, n))
    sizes, offsets, signals = _table([[rows, n]] * world), _table([[rows, 0], [0, 0]]), _table([1, 0])
    flags = torch.zeros(world, dtype=torch.int64, device="cuda")
    c = torch.zeros(m, n, dtype=torch.bfloat16, device="cuda")

    def run(sizes=sizes, a=a, n=n):
        c.zero_()
        flags.fill_(form == "consumer")
        if form == "direct":
            gemm_rs_producer_persistent(a, b, list(c.view(world, rows, n)), sizes, offsets, signals, world, world, 64, 128, 128, 64, 8)
        elif form == "producer":
            gemm_producer(a, b, c, flags, sizes, offsets, signals, 64, 128, 128, 64, 8, cum_tiles=m * n)
            assert flags.tolist() == [1] * world
        else:
            gemm_consumer(a, b, c, flags, sizes, offsets, signals, world, 64, 128, 128, 64, 8, cum_tiles=m * n)
        return c.clone()

    want = a.float() @ b.float().T
    if form == "direct":                       # wave 0 (the second half) goes to rank 1, wave 1 to rank 0: in place
        want = want.view(world, rows, n).reshape(m, n)
    return run, want, sizes, a, template_remote if form == "direct" else template


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["consumer", "producer", "direct"])
def test_gemm_second_launch(hip, monkeypatch, form):
    from syncopate_amd.computation._launch import check_status

    run, want, sizes, a, module = _gemm_case(form)
    first = run()
    check_status()
    # one rounding of the result (2^-9 relative), sums in 32 bits
    assert (first.float() - want).abs().max() <= 4e-3 * want.abs().max()
    general, convert = [], module.as_device_table
    monkeypatch.setattr(module, "as_device_table", lambda *args: general.append(1) or convert(*args))
    for _ in range(40):                        # the pool of counters is filled again on the way
        again = run()
    check_status()
    assert torch.equal(again, first) and not general
    # a write into a table: read and checked again, and refused if it does not fit any more
    sizes.add_(0)
    assert torch.equal(run(), first) and general
    general.clear()
    assert torch.equal(run(), first) and not general
    # a subclass, an operand elsewhere, other tables with the same contents, a table that no longer fits
    assert torch.equal(run(a=torch.nn.Parameter(a, requires_grad=False)), first) and not general
    assert torch.equal(run(a=torch.cat([a, a])[:len(a)]), first) and not general
    assert torch.equal(run(sizes=sizes.clone()), first) and general
    with pytest.raises(Exception):
        run(a=a.cpu())
    sizes[0, 0] = 64
    with pytest.raises(_lib.SyncopateHipError):
        run()


@pytest.mark.gpu
@pytest.mark.parametrize("launcher", ["gemm_consumer", "gemm_producer", "gemm_rs_producer_persistent", "gemm_remote", "gemm_splitk",
                                      "gemm_ag_direct_read", "ring_reduce", "attention_forward"])
def test_given_stream(hip, launcher):
    """Calls with `stream`, after one without and again on the same operands: ordered with what was queued there in front of them,
    the operand that arrives late and the zeroing of a C that is added to."""
    from syncopate_amd.computation import attn, gemm, reduce
    from syncopate_amd.computation._launch import check_status

    g = torch.Generator(device="cuda").manual_seed(3)
    randn = lambda *shape: (0.1 * torch.randn(shape, device="cuda", generator=g)).bfloat16()
    m, n, k = 512, 512, 128
    a, b, c = randn(m, k), randn(n, k), torch.zeros(m, n, dtype=torch.bfloat16, device="cuda")
    sizes, offsets, waves = _table([[256, n]] * 2), _table([[0, 0], [256, 0]]), _table([0, 1])
    flags = torch.ones(2, dtype=torch.int64, device="cuda")
    halves, late, out = list(c.view(2, 256, n)), a, c
    if launcher == "gemm_consumer":
        call = lambda **kw: gemm.gemm_consumer(a, b, c, flags, sizes, offsets, waves, 2, 64, 128, 128, 64, 8, cum_tiles=m * n, **kw)
    elif launcher == "gemm_producer":
        call = lambda **kw: gemm.gemm_producer(a, b, c, flags, sizes, offsets, waves, 64, 128, 128, 64, 8, cum_tiles=m * n, **kw)
    elif launcher == "gemm_rs_producer_persistent":
        call = lambda **kw: gemm.gemm_rs_producer_persistent(a, b, halves, sizes, offsets, waves, 2, 2, 64, 128, 128, 64, 8, **kw)
    elif launcher == "gemm_remote":
        rows = _table([[0, 0], [0, 0]])
        call = lambda **kw: gemm.gemm_remote(a, b, halves, 64, 128, 128, 64, 8, cur_wave_sizes=sizes, wave_offsets=offsets, M=m,
                                             target_rank=waves, dst_offsets=rows, **kw)
    elif launcher == "gemm_splitk":
        boxes = _table([[m, n, 64]] * 2), _table([[0, 0, 0], [0, 0, 64]])
        call = lambda **kw: gemm.gemm_splitk(a, b, c, 2, 64, 128, 128, 64, 8, cur_wave_sizes=boxes[0], wave_offsets=boxes[1],
                                             cum_tiles=2 * m * n, **kw)
    elif launcher == "gemm_ag_direct_read":
        call = lambda **kw: gemm.gemm_ag_direct_read(list(a.view(2, 256, k)), b, c, sizes, offsets, waves, 2, 2, 64,
                                                     BLOCK_SIZE_N=128, **kw)
    elif launcher == "ring_reduce":
        late, out = randn(2, 256, n), torch.zeros(256, n, dtype=torch.bfloat16, device="cuda")
        call = lambda **kw: reduce.ring_reduce(late, out, c, 0, **kw)
    else:
        q, late, out = randn(1, 1, 256, 128), randn(1, 1, 256, 128), torch.zeros(1, 1, 256, 128, dtype=torch.bfloat16, device="cuda")
        tables = dict(wave_offsets=_table([[0, 0, 0, 0]]), wave_sizes=_table([[1, 1, 256, 256]]), cum_wave_sizes=_table([256]),
                      signal_offsets=_table([0]), cum_tiles=256)
        call = lambda **kw: attn.attention_forward(q, late, late, 0.1, signal_ptr=flags, output_buffer=out, **tables, **kw)
    call()
    torch.cuda.synchronize()
    want, real, lib = out.clone(), late.clone(), _lib.load()
    assert want.abs().max() > 0 or launcher == "ring_reduce"
    side = torch.cuda.Stream()
    for _ in range(3):
        late.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            _lib.check("syn_delay_us", lib.syn_delay_us(5000, _lib.stream_handle(side)))
            late.copy_(real)
            out.zero_()
        call(stream=side)
        side.synchronize()
        check_status()
        assert torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("differ", ["buffers", "programs", "tile", "stream"])
def test_launches_in_turn_on_one_set_of_tables(hip, monkeypatch, differ):
    """Launches that share their tables and differ in something else are known side by side."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.gemm import gemm_consumer, gemm_rs_producer_persistent, template, template_remote

    m, n, k = 512, 512, 192
    g = torch.Generator(device="cuda").manual_seed(3)
    a, b = ((0.1 * torch.randn(s, k, device="cuda", generator=g)).bfloat16() for s in (m, n))
    sizes, offsets, waves = _table([[256, n]] * 2), _table([[0, 0], [256, 0]]), _table([0, 1])
    flags = torch.ones(2, dtype=torch.int64, device="cuda")
    results = [torch.zeros(2, 256, n, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    bound, streams = [list(c) for c in results], [torch.cuda.current_stream(), torch.cuda.Stream()]
    general, convert = [], template.as_device_table
    for module in (template, template_remote):
        monkeypatch.setattr(module, "as_device_table", lambda *args: general.append(1) or convert(*args))
    want = (a.float() @ b.float().T).view(2, 256, n)
    for turn in range(6):
        which = turn % 2
        into, programs, bn = which if differ == "buffers" else 0, 48 + 16 * (differ == "programs" and which), 128 << (differ == "tile" and which)
        results[into].zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[which if differ == "stream" else 0]):
            gemm_rs_producer_persistent(a, b, bound[into], sizes, offsets, waves, 2, 2, programs, 128, bn, 64, 8)
            torch.cuda.synchronize()
            # one rounding of the result (2^-9 relative), sums in 32 bits
            assert (results[into].float() - want).abs().max() <= 4e-3 * want.abs().max()
            results[into].zero_()
            gemm_consumer(a, b, results[into].view(m, n), flags, sizes, offsets, waves, 2, programs, 128, bn, 64, 8, cum_tiles=m * n)
            torch.cuda.synchronize()
            assert (results[into].float() - want).abs().max() <= 4e-3 * want.abs().max()
        if turn == 1:
            general.clear()
    check_status()
    assert not general


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["direct", "split k"])
def test_captured_behind_a_launch_on_another_stream(hip, form):
    """What an eager launch has prepared serves the capture, whose stream is another one; replays among eager launches."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.gemm import gemm_rs_producer_persistent, gemm_splitk

    m, n, k = 512, 512, 128
    g = torch.Generator(device="cuda").manual_seed(3)
    a, b = ((0.1 * torch.randn(s, k, device="cuda", generator=g)).bfloat16() for s in (m, n))
    c = torch.zeros(m, n, dtype=torch.bfloat16, device="cuda")
    sizes, offsets, waves = _table([[256, n]] * 2), _table([[0, 0], [256, 0]]), _table([0, 1])
    boxes, halves = (_table([[m, n, 64]] * 2), _table([[0, 0, 0], [0, 0, 64]])), list(c.view(2, 256, n))

    def launch():
        c.zero_()
        if form == "direct":
            gemm_rs_producer_persistent(a, b, halves, sizes, offsets, waves, 2, 2, 64, 128, 128, 64, 8)
        else:
            gemm_splitk(a, b, c, 2, 64, 128, 128, 64, 8, cur_wave_sizes=boxes[0], wave_offsets=boxes[1], cum_tiles=2 * m * n)

    launch()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch()
    for turn in range(4):
        a.mul_(-1)
        launch()
        want = c.clone()
        c.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        check_status()
        assert torch.equal(c, want) and want.any()


@pytest.mark.gpu
@pytest.mark.parametrize("warm", [True, False])
def test_captured_launch_has_tables_of_its_own(hip, monkeypatch, warm):
    """The tables of waves that wait for nothing, in a captured launch: not those that eager launches share and a record keeps, whether
    the captured number of waves was seen before or not."""
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.gemm import gemm_remote, template_remote

    m, n, k, waves = 512, 512, 128, 4 if warm else 2
    g = torch.Generator(device="cuda").manual_seed(3)
    a, b = ((0.1 * torch.randn(s, k, device="cuda", generator=g)).bfloat16() for s in (m, n))
    c = torch.zeros(m, n, dtype=torch.bfloat16, device="cuda")
    sizes, offsets = _table([[m // waves, n]] * waves), _table([[i * m // waves, 0] for i in range(waves)])
    owners, bound = _table([0] * waves), [c]
    launch = lambda: gemm_remote(a, b, bound, 64, 128, 128, 64, 8, cur_wave_sizes=sizes, wave_offsets=offsets, M=m, target_rank=owners,
                                 dst_offsets=offsets)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        launch()                                         # prepared, and a record of this stream
        launch()
        torch.cuda.synchronize()
        if not warm:
            monkeypatch.setattr(template_remote, "_NO_SIGNALS", {})
        kept = dict(template_remote._NO_SIGNALS)
        made, full = [], torch.full
        monkeypatch.setattr(torch, "full", lambda shape, *args, **kw: made.append(shape) or full(shape, *args, **kw))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            launch()
        assert made == [(waves,)] and template_remote._NO_SIGNALS == kept
    a.mul_(-1)
    want = a.float() @ b.float().T
    for _ in range(3):
        c.zero_()
        graph.replay()
        torch.cuda.synchronize()
        check_status()
        # one rounding of the result (2^-9 relative), sums in 32 bits
        assert (c.float() - want).abs().max() <= 4e-3 * want.abs().max()
        launch()


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["consumer", "direct"])
def test_another_rule_for_the_tile_is_asked(hip, form):
    """Rules made and dropped one after the other, as a caller's own may be: each is asked, wherever it lies in memory."""
    from syncopate_amd.computation._launch import check_status

    run, want, _, _, module = _gemm_case(form)
    rule, asked, places = module.choose_kernel_tile, [], set()
    try:
        for turn in range(4):
            module.choose_kernel_tile = lambda *args, **kw: asked.append(turn) or rule(*args, **kw)
            places.add(id(module.choose_kernel_tile))
            for _ in range(2):
                assert (run().float() - want).abs().max() <= 4e-3 * want.abs().max()
    finally:
        module.choose_kernel_tile = rule
    check_status()
    assert asked == [0, 1, 2, 3] and len(places) == 4


@pytest.mark.gpu
def test_first_launches_inside_inference_mode(hip):
    """The pools of zeroed words, of the native launches and of the launchers, are made inside the mode and filled again outside."""
    from syncopate_amd.computation._launch import ZERO_POOL_SLICES, check_status, zeroed_int32

    run, want, *_ = _gemm_case("producer")
    with torch.cuda.stream(torch.cuda.Stream()):
        torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
        run()                                            # (remembers the tables; a pool of this stream is still to be made)
        with torch.inference_mode():
            assert (run().float() - want).abs().max() <= 4e-3 * want.abs().max()
        for _ in range(20):
            assert (run().float() - want).abs().max() <= 4e-3 * want.abs().max()
        with torch.inference_mode():
            zeroed_int32((7,), torch.device("cuda", 0))
        for _ in range(ZERO_POOL_SLICES + 1):
            words = zeroed_int32((7,), torch.device("cuda", 0))
            assert not words.any()
            words.fill_(1)
    check_status()


@pytest.mark.gpu
def test_threads_and_streams(hip):
    """Producers of two threads on streams of their own, more launches than a pool of counters has areas."""
    from syncopate_amd.computation._launch import check_status

    failed = []

    def work():
        try:
            stream = torch.cuda.Stream()
            stream.wait_stream(torch.cuda.default_stream())
            with torch.cuda.stream(stream):
                run, want, *_ = _gemm_case("producer")
                for _ in range(50):
                    assert (run().float() - want).abs().max() <= 4e-3 * want.abs().max()
            stream.synchronize()
        except BaseException as exc:                                    # noqa: BLE001
            failed.append(exc)

    threads = [threading.Thread(target=work) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    check_status()
    assert not failed, failed


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
@pytest.mark.parametrize("form", ["explicit", "auto", "causal auto", "producer"])
def test_attention_second_launch(hip, monkeypatch, form, layout):
    from oracle import numerics
    from syncopate_amd.computation._launch import check_status
    from syncopate_amd.computation.attn import attention_forward, template

    H, S, waves = 2, 512, 2
    causal, producer = form == "causal auto", form == "producer"
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(1, H, S, 128, generator=g).half() for _ in range(3))
    lay = (lambda t: t.cuda()) if layout == "bhsd" else (lambda t: t.permute(0, 2, 1, 3).contiguous().cuda())
    qd, kd, vd = lay(q), lay(k), lay(v)
    split_q = producer
    offsets = _table([[0, 0, i * 256 if split_q else 0, 0 if split_q else i * 256] for i in range(waves)])
    sizes = _table([[1, H, 256 if split_q else S, S if split_q else 256]] * waves)
    rows = H * (256 if split_q else S)
    cums, signals = _table([rows, 2 * rows]), _table([0, 1])
    flags = torch.ones(waves, dtype=torch.int64, device="cuda")
    counters = torch.zeros(waves, dtype=torch.int32, device="cuda") if producer else None

    def run(scale=0.1, **kw):
        if producer:
            flags.zero_()
            counters.zero_()
        got = attention_forward(qd, kd, vd, scale, wave_offsets=offsets, wave_sizes=sizes, cum_wave_sizes=cums,
                                signal_ptr=flags, signal_offsets=signals, NUM_WAVES=waves, cum_tiles=2 * rows, causal=causal,
                                layout=layout, counter_ptr=counters, form="auto" if "auto" in form else "explicit", **kw)
        check_status()
        assert flags.tolist() == [1] * waves and (not producer or counters.tolist() == [rows // 128] * waves)
        return got

    def near(out, scale=0.1):
        out = (out if layout == "bhsd" else out.permute(0, 2, 1, 3)).float().cpu()
        want = numerics.sdpa_fp32(q, k, v, scale, causal=causal)
        # roundings of the result, of the probabilities and of a merged result, 2^-12 each relative to the largest; four times that
        return (out - want).abs().max() <= 4e-3 * want.abs().max()

    first, lse = run(return_lse=True)
    assert near(first) and near(run())         # without and with lse are two things to remember
    general, convert = [], template.as_device_table
    monkeypatch.setattr(template, "as_device_table", lambda *args: general.append(1) or convert(*args))
    for _ in range(20):
        assert near(run())
    assert near(run(0.3), 0.3)
    out = torch.full_like(qd, float("nan"))
    assert run(out=out) is out and near(out)
    again, lse2 = run(return_lse=True)
    assert near(again) and (lse2 - lse).abs().max() <= 1e-4 and not general
    sizes.add_(0)
    assert near(run()) and general
    general.clear()
    with pytest.raises(ValueError):
        run(out=torch.empty(1, H, S, 64, device="cuda", dtype=torch.half))
    sizes[0, 2] = 192
    with pytest.raises(Exception):
        run()


@pytest.mark.gpu
@pytest.mark.parametrize("acc_mode", ["dtype", "fp32"])
def test_reduce_is_launched_or_refused(hip, monkeypatch, acc_mode):
    from syncopate_amd.computation import reduce as module

    g = torch.Generator(device="cuda").manual_seed(1)
    received, local = (torch.randn(s, device="cuda", generator=g).half() for s in ((3, 40, 64), (120, 64)))
    out = torch.empty(40, 64, dtype=torch.half, device="cuda")
    seen, ask = [], module.require_cuda
    monkeypatch.setattr(module, "require_cuda", lambda *args: seen.append(1) or ask(*args))
    assert module.ring_reduce(received, out, local, 1, acc_mode=acc_mode) is out and not seen
    want = local[40:80].float()
    for i in (2, 0):
        want = want + received[i].float()
        want = want.half().float() if acc_mode == "dtype" else want
    assert torch.equal(out, want.half())
    with pytest.raises(ValueError):
        module.ring_reduce(received, out, local.t().contiguous().t(), 1, acc_mode=acc_mode)
    with pytest.raises(TypeError):
        module.ring_reduce(received, out, local.float(), 1, acc_mode=acc_mode)
    with pytest.raises(_lib.SyncopateHipError):
        module.ring_reduce(received, out, local, 3, acc_mode=acc_mode)


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 3, 64, 341])
def test_tables_are_read_at_their_place_in_the_stream(hip, rows):
    native = _lib.native()
    g = torch.Generator(device="cuda").manual_seed(rows)
    offsets, sizes = (torch.randint(-9, 2 ** 30, (4 * rows,), device="cuda", generator=g, dtype=torch.int32) for _ in range(2))
    cums, signals = (torch.randint(-9, 2 ** 30, (rows,), device="cuda", generator=g, dtype=torch.int32) for _ in range(2))
    for stream in (torch.cuda.current_stream(), torch.cuda.Stream()):
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            for round in range(12):
                torch.cuda._sleep(100_000 if round % 4 else 20_000_000)      # behind work that takes 40 us, or 10 ms
                cums.add_(1)
                got = native.read_tables(offsets.view(-1, 4), sizes, cums, signals)
                want = torch.cat([offsets, sizes, cums, signals]).cpu()
                assert got == want.numpy().tobytes()
        stream.synchronize()
    assert native.read_tables(offsets, sizes, cums, signals.long()) is None
    assert native.read_tables(offsets, sizes, cums, signals.cpu()) is None
    assert native.read_tables(offsets.view(-1, 2).t(), sizes) is None and native.read_tables() is None
    assert native.read_tables(torch.cat([offsets] * 8192)[:8192], sizes, cums, signals) is None if rows >= 3 else True
