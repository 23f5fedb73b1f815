"""The HIP local reduction (the reduce stage of the failure-detecting all-reduce) on the GPU.

Bits equal to the oracle's ordered fp32 sum (core/everserve/reference/arith/ops.py:63-73) at the
reference's sizes {16384, 3000, 2} (core/tests/test_slot_kernel.py:40) and at C5 (8 buffers of
256 x 8192); the order-sensitive inputs of core/tests/test_slot_kernel.py:50-55; and the bounded
wait: a stalled flag ends in a timeout naming that row, the host's ABORT word releases the wait,
the LATE word names the stalled row while the wait passes BOUND and is cleared after, and a flag
that arrives late (host-mapped, written by the host mid-wait) completes the call normally. A
workgroup that finds members missing loads the others before it waits (early start): members
that arrive late in the middle of the order, over several passes and an element tail, and one
that never arrives, are summed exactly as a call that waited first. Every wait in these tests is
bounded by the kernel's own timeout.
"""

import ctypes
import threading
import time

import numpy as np
import pytest
import torch

import oracle
from everserve_amd.kernels import REDUCE_STATE_WORDS
from tests.cases import bf16_tensor, bits, special_members

pytestmark = pytest.mark.gpu

MAXW = 8
ABORT, LATE, BOUND = 1, 11, 12


def bf16_input(seed: int, n: int) -> torch.Tensor:
    g = torch.Generator().manual_seed(seed)
    return torch.randn(n, generator=g).to(torch.bfloat16)


class Ctrl:
    """One control row of 16 int64 words in pinned, coherent host memory mapped into the GPU."""

    def __init__(self, ext):
        self.ext = ext
        self.host, self.dev = ext.host_alloc_mapped(16 * 8)
        self.words = (ctypes.c_int64 * 16).from_address(self.host)

    def close(self):
        self.ext.host_free(self.host)


def named(ctrl: Ctrl, rows_mask: int, within_s: float = 2.0) -> bool:
    """Poll the host-mapped LATE word until it names every row of ``rows_mask``: the call has
    found those members missing and is waiting for them (past BOUND), so their flags, written
    after this, arrive during its wait rather than before its launch."""
    deadline = time.perf_counter() + within_s
    while time.perf_counter() < deadline:
        if int(ctrl.words[LATE]) & rows_mask == rows_mask:
            return True
        time.sleep(0.0002)
    return False


class Members:
    """k member buffers in HBM, their flags, the order, and the call's state."""

    def __init__(self, inputs: dict[int, torch.Tensor], order: list[int]):
        self.bufs_t = {r: x.cuda() for r, x in inputs.items()}
        table = [0] * MAXW
        for r, t in self.bufs_t.items():
            table[r] = t.data_ptr()
        self.bufs = torch.tensor(table, dtype=torch.long, device="cuda")
        self.flags = torch.zeros(MAXW, dtype=torch.long, device="cuda")
        self.order = torch.tensor([len(order), *order] + [0] * (MAXW - len(order)),
                                  dtype=torch.int32, device="cuda")
        self.state = torch.zeros(REDUCE_STATE_WORDS, dtype=torch.long, device="cuda")
        n = next(iter(inputs.values())).numel()
        self.out = torch.empty(n, dtype=torch.bfloat16, device="cuda")

    def publish(self, epoch: int, rows=None):
        rows = rows if rows is not None else list(self.bufs_t)
        f = self.flags.cpu()
        for r in rows:
            f[r] = epoch
        self.flags.copy_(f)

    def status(self):
        s = int(self.state[0].item()) & 0xFFFFFFFFFFFFFFFF
        return s >> 16, (s >> 8) & 0xFF, s & 0xFF


@pytest.mark.parametrize("n", [16384, 3000, 2, 8 * 256 * 2 + 5, 40960, 65536])
@pytest.mark.parametrize("order", [[0, 1, 2], [2, 0, 1], [5, 3, 7, 0, 1, 6, 2, 4]])
def test_the_sum_is_the_ordered_fp32_sum_bit_for_bit(ext, n, order):
    inputs = {r: bf16_input(1000 * r + n, n) for r in order}
    m = Members(inputs, order)
    m.publish(epoch=1)
    ext.local_reduce(m.bufs, m.flags, m.order, m.out, 1, 10**9, 0, m.state)
    torch.cuda.synchronize()
    want = oracle.member_sum([bits(inputs[r]) for r in order])
    assert np.array_equal(bits(m.out), want)
    assert m.status() == (1, 0, 0)
    assert not m.state[1:].any()  # the kernel's counters are back at zero


@pytest.mark.parametrize("vectors", [1, 255, 256, 257, 9000, 70_000, 140_000])
@pytest.mark.parametrize("tail", [1, 4, 7])
@pytest.mark.parametrize("absent", [None, 3])
def test_the_elements_past_the_last_vector(ext, vectors, tail, absent):
    """1 to 7 elements past the vectors, in every counting mode and vector width, with every
    member in and with one that never comes (it sums as zeros)."""
    n, order = 8 * vectors + tail, [4, 3, 0, 6]
    inputs = {r: bf16_input(77 * r + n, n) for r in order}
    m = Members(inputs, order)
    m.publish(epoch=5, rows=[r for r in order if r != absent])
    ext.local_reduce(m.bufs, m.flags, m.order, m.out, 5, 10**9 if absent is None else 10**6, 0,
                     m.state)
    torch.cuda.synchronize()
    want = oracle.member_sum([bits(inputs[r]) * (r != absent) for r in order])
    assert np.array_equal(bits(m.out), want)
    assert m.status() == ((5, 0, 0) if absent is None else (5, 2, 1 << absent))
    assert not m.state[1:].any()


@pytest.mark.parametrize("order", [[2], [5, 0], [1, 7, 4], [3, 0, 6, 2]])
@pytest.mark.parametrize("passes", [0.6, 1.3, 2.6, 3.5, 4.2, 8.1])
def test_few_members_take_several_passes_at_once(ext, order, passes):
    """One to four members over part of a pass, one, and group edges (two and four passes at a
    time, and the passes past which four members go one at a time), with a member that is late
    from the start in one more call: the ordered fp32 sum bit for bit."""
    n = int(passes * (1 << 21)) + 3
    inputs = {r: bf16_input(40 + r, n) for r in order}
    m = Members(inputs, order)
    m.publish(epoch=2)
    ext.local_reduce(m.bufs, m.flags, m.order, m.out, 2, 10**9, 0, m.state)
    torch.cuda.synchronize()
    assert np.array_equal(bits(m.out), oracle.member_sum([bits(inputs[r]) for r in order]))
    assert m.status() == (2, 0, 0) and not m.state[1:].any()
    m.publish(epoch=3, rows=order[:-1])  # the last member never comes
    ext.local_reduce(m.bufs, m.flags, m.order, m.out, 3, 10**6, 0, m.state)
    torch.cuda.synchronize()
    want = oracle.member_sum([bits(inputs[r]) * (r != order[-1]) for r in order])
    assert np.array_equal(bits(m.out), want)
    assert m.status() == (3, 2, 1 << order[-1])


@pytest.mark.parametrize("order", [[3, 0], [2, 6, 0, 5], [5, 3, 7, 0, 1, 6, 2, 4]])
@pytest.mark.parametrize("n", [8 * 70_000 + 5, 8 * 140_000 + 1, 3_000_007])
def test_a_flag_that_lands_while_the_workgroups_start(ext, order, n):
    """A member's flag is written 0 to 30 us after the launch call, and every other time with
    another stream's copy on the CUs, so that it lands between the workgroups' first reads of the
    flags: some find the member in and some start early (two launches of three; in one of forty
    the last workgroup starts early and the first does not). Whatever the mix, every element is
    written, those past the last vector too: ``out`` is filled with a pattern first."""
    flags_host, flags_dev = ext.host_alloc_mapped(MAXW * 8)
    try:
        words = (ctypes.c_int64 * MAXW).from_address(flags_host)
        inputs = {r: bf16_input(90 + r, n) for r in order}
        m = Members(inputs, order)
        want = torch.from_numpy(oracle.member_sum([bits(inputs[r]) for r in order])
                                .view(np.int16)).cuda()
        unwritten = 0x7F5A  # a NaN no rounding gives
        late, side = order[1], torch.cuda.Stream()
        busy = torch.zeros((2, 16 << 20), dtype=torch.int32, device="cuda")
        for i in range(120):
            epoch = i + 1
            m.out.view(torch.int16).fill_(unwritten)
            for r in order:
                words[r] = epoch - 1 if r == late else epoch
            torch.cuda.synchronize()
            if i % 2:
                with torch.cuda.stream(side):
                    busy[0].copy_(busy[1])
            ext.local_reduce(m.bufs, flags_dev, m.order, m.out, epoch, 3_000_000_000, 0, m.state)
            release = time.perf_counter_ns() + (i // 2) * 500
            while time.perf_counter_ns() < release:
                pass
            words[late] = epoch
            torch.cuda.synchronize()
            got = m.out.view(torch.int16)
            wrong = torch.nonzero(got != want)
            assert not wrong.numel(), (i, wrong.flatten().tolist()[:8], got[-8:].tolist())
            assert m.status() == (epoch, 0, 0) and not m.state[1:].any()
    finally:
        ext.host_free(flags_host)


@pytest.mark.parametrize("order", [[2], [5, 0], [1, 7, 4], [3, 0, 6, 2]])
@pytest.mark.parametrize("n", [(1 << 20) + 11, int(2.6 * (1 << 21)) + 3])
def test_few_members_one_of_which_arrives_mid_wait(ext, order, n):
    """One to four members, the last of which is named late and then arrives: part of a pass and
    several, with elements past the last vector."""
    flags_host, flags_dev = ext.host_alloc_mapped(MAXW * 8)
    ctrl = Ctrl(ext)
    try:
        words = (ctypes.c_int64 * MAXW).from_address(flags_host)
        inputs = {r: bf16_input(20 + r, n) for r in order}
        m = Members(inputs, order)
        m.out.zero_()
        for r in order:
            words[r] = 0 if r == order[-1] else 4
        torch.cuda.synchronize()
        ctrl.words[BOUND] = 100_000
        ext.local_reduce(m.bufs, flags_dev, m.order, m.out, 4, 3_000_000_000, ctrl.dev, m.state)
        try:
            waited = named(ctrl, 1 << order[-1])
        finally:
            words[order[-1]] = 4
        torch.cuda.synchronize()
        assert waited, "the call never named the last member: it did not wait for it"
        assert np.array_equal(bits(m.out), oracle.member_sum([bits(inputs[r]) for r in order]))
        assert m.status() == (4, 0, 0) and not m.state[1:].any()
        assert int(ctrl.words[LATE]) == 0
    finally:
        ctrl.close()
        ext.host_free(flags_host)


@pytest.mark.parametrize("n", [3 * (1 << 20) + 5, 6 * (1 << 20)])
def test_calls_past_the_resident_grid_take_several_passes(ext, n):
    """Past 2 Mi elements the 4-vector kernel's grid stays at 256 workgroups, one a CU with the
    counting wave beside the payload's, so each workgroup takes several passes: the sum is still
    the ordered fp32 sum bit for bit, the outcome is counted once, the counters end at zero."""
    order = [6, 1, 4, 0, 3, 7, 2, 5]
    inputs = {r: bf16_input(300 + r, n) for r in order}
    m = Members(inputs, order)
    m.publish(epoch=2)
    ext.local_reduce(m.bufs, m.flags, m.order, m.out, 2, 10**9, 0, m.state)
    torch.cuda.synchronize()
    want = oracle.member_sum([bits(inputs[r]) for r in order])
    assert np.array_equal(bits(m.out), want)
    assert m.status() == (2, 0, 0)
    assert not m.state[1:].any()


def test_the_order_of_the_sum_shows_and_is_kept(ext):
    n = 16384
    g = torch.Generator().manual_seed(7)
    big = torch.randn(n, generator=g) * 2.0**20
    small = torch.randn(n, generator=g) * 2.0**-6
    inputs = {0: big.to(torch.bfloat16), 1: small.to(torch.bfloat16), 2: (-big).to(torch.bfloat16)}
    in_rank = oracle.member_sum([bits(inputs[r]) for r in (0, 1, 2)])
    in_rows = oracle.member_sum([bits(inputs[r]) for r in (0, 2, 1)])
    assert not np.array_equal(in_rank, in_rows), "the inputs must make the order show"
    for order, want in (([0, 1, 2], in_rank), ([0, 2, 1], in_rows)):
        m = Members(inputs, order)
        m.publish(epoch=9)
        ext.local_reduce(m.bufs, m.flags, m.order, m.out, 9, 10**9, 0, m.state)
        torch.cuda.synchronize()
        assert np.array_equal(bits(m.out), want)


def test_c5_eight_buffers_of_256_by_8192(ext):
    n = 256 * 8192
    order = list(range(8))
    inputs = {r: bf16_input(5 + r, n) for r in order}
    m = Members(inputs, order)
    m.publish(epoch=3)
    for _ in range(3):  # replays: the state's counters reset themselves
        ext.local_reduce(m.bufs, m.flags, m.order, m.out, 3, 10**9, 0, m.state)
    torch.cuda.synchronize()
    want = oracle.member_sum([bits(inputs[r]) for r in order])
    assert np.array_equal(bits(m.out), want)
    assert m.status() == (3, 0, 0)


@pytest.mark.parametrize("n", [256 * 8192, 81920, 65536, 10000, 2048])
def test_a_stalled_flag_ends_in_a_timeout_that_names_it(ext, n):
    """At C5 (256 workgroups of 4 vectors a thread) and 81920 elements (40 workgroups of 1), both
    counted in two levels; 65536 (32 workgroups) and 10000 (5), counted in the top word; and 2048
    (one, nothing counted): the outcome word names the stalled row each way."""
    order = list(range(8))
    inputs = {r: bf16_input(5 + r, n) for r in order}
    m = Members(inputs, order)
    m.publish(epoch=4)
    m.publish(epoch=3, rows=[3])  # row 3's flag stays at epoch - 1
    t0 = time.perf_counter()
    ext.local_reduce(m.bufs, m.flags, m.order, m.out, 4, 1_000_000, 0, m.state)  # 1 ms
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    assert m.status() == (4, 2, 1 << 3)
    want, reason, late = oracle.reduce_protocol({r: bits(x) for r, x in inputs.items()},
                                                {r: (3 if r == 3 else 4) for r in order}, order, 4)
    assert (reason, late) == (2, 1 << 3)
    assert np.array_equal(bits(m.out), want)
    assert elapsed < 2.0, elapsed


def test_the_abort_word_releases_the_wait(ext):
    ctrl = Ctrl(ext)
    try:
        inputs = {r: bf16_input(r, 4096) for r in range(3)}
        m = Members(inputs, [0, 1, 2])
        m.publish(epoch=6, rows=[0, 2])  # row 1 never arrives
        t0 = time.perf_counter()
        ext.local_reduce(m.bufs, m.flags, m.order, m.out, 6, 5_000_000_000, ctrl.dev, m.state)
        time.sleep(0.05)
        ctrl.words[ABORT] = 1
        torch.cuda.synchronize()
        elapsed = time.perf_counter() - t0
        assert m.status() == (6, 1, 1 << 1)
        assert elapsed < 4.0, elapsed  # well inside the 5 s timeout
    finally:
        ctrl.close()


def test_the_late_word_names_the_stalled_row_then_clears(ext):
    ctrl = Ctrl(ext)
    try:
        inputs = {r: bf16_input(r, 65536) for r in range(4)}
        m = Members(inputs, [0, 1, 2, 3])
        m.publish(epoch=2, rows=[0, 1, 3])
        ctrl.words[BOUND] = 1_000_000  # name after 1 ms
        seen = set()
        ext.local_reduce(m.bufs, m.flags, m.order, m.out, 2, 300_000_000, ctrl.dev, m.state)
        deadline = time.perf_counter() + 0.25
        while time.perf_counter() < deadline:
            seen.add(int(ctrl.words[LATE]))
            time.sleep(0.001)
        torch.cuda.synchronize()
        assert (1 << 2) in seen, seen
        assert seen <= {0, 1 << 2}, seen
        assert int(ctrl.words[LATE]) == 0  # cleared by the last workgroup that named
        assert m.status() == (2, 2, 1 << 2)
    finally:
        ctrl.close()


def test_a_flag_that_arrives_late_completes_the_call(ext):
    flags_host, flags_dev = ext.host_alloc_mapped(MAXW * 8)
    try:
        words = (ctypes.c_int64 * MAXW).from_address(flags_host)
        inputs = {r: bf16_input(40 + r, 30000) for r in range(3)}
        m = Members(inputs, [1, 0, 2])
        for r in (0, 1):
            words[r] = 12
        ext.local_reduce(m.bufs, flags_dev, m.order, m.out, 12, 3_000_000_000, 0, m.state)
        time.sleep(0.02)
        words[2] = 12  # the last member's payload was in place all along; now its flag
        torch.cuda.synchronize()
        assert m.status() == (12, 0, 0)
        want = oracle.member_sum([bits(inputs[r]) for r in (1, 0, 2)])
        assert np.array_equal(bits(m.out), want)
    finally:
        ext.host_free(flags_host)


@pytest.mark.parametrize("n", [256 * 8192, 2 * 1024 * 256 * 4 * 8 + 8 * 3 + 5])
def test_members_that_arrive_late_in_the_middle_of_the_order(ext, n):
    """Rows 0 and 6 sit mid-order and arrive one after the other while the call waits. A
    workgroup loads the members already in before it waits, so the late ones are summed in their
    order positions among them. The second size takes three passes of the grid and ends in an
    element tail."""
    flags_host, flags_dev = ext.host_alloc_mapped(MAXW * 8)
    ctrl = Ctrl(ext)
    try:
        words = (ctypes.c_int64 * MAXW).from_address(flags_host)
        order = [5, 3, 7, 0, 1, 6, 2, 4]
        inputs = {r: bf16_input(60 + r, n) for r in order}
        m = Members(inputs, order)
        for r in order:
            words[r] = 0 if r in (0, 6) else 9
        ctrl.words[BOUND] = 100_000  # name the rows still awaited after 0.1 ms of waiting
        ext.local_reduce(m.bufs, flags_dev, m.order, m.out, 9, 3_000_000_000, ctrl.dev, m.state)
        try:
            waited = named(ctrl, (1 << 0) | (1 << 6))
            words[6] = 9
            time.sleep(0.01)
        finally:
            words[6] = words[0] = 9
        torch.cuda.synchronize()
        assert waited, "the call never named rows 0 and 6 as late: it did not wait for them"
        assert m.status() == (9, 0, 0)
        assert int(ctrl.words[LATE]) == 0
        want = oracle.member_sum([bits(inputs[r]) for r in order])
        assert np.array_equal(bits(m.out), want)
    finally:
        ctrl.close()
        ext.host_free(flags_host)


@pytest.mark.parametrize("n", [2048, 2048 + 8, 32 * 256 * 8, 32 * 256 * 8 + 8,
                               256 * 256 * 8, 256 * 256 * 8 + 13, 2 * 256 * 256 * 8,
                               2 * 256 * 256 * 8 + 8 * 5 + 3])
def test_grids_at_the_launch_thresholds(ext, n):
    """The launch takes 1, 2 or 4 vectors a thread, the fewest that keep the grid within 256
    workgroups, and counts completion by the grid: not at all in a grid of one, in the top word
    up to 32 workgroups, in two levels past that. These sizes sit on either side of each switch:
    1 | 2 and 32 | 33 workgroups of 1 vector a thread, then the 1 -> 2 and 2 -> 4 vector
    switches. At each, every member in, then one of them arriving while the call waits, summed as
    the oracle does, with the counting words back at zero."""
    flags_host, flags_dev = ext.host_alloc_mapped(MAXW * 8)
    ctrl = Ctrl(ext)
    try:
        words = (ctypes.c_int64 * MAXW).from_address(flags_host)
        order = [6, 1, 4, 0, 7, 2, 5, 3]
        inputs = {r: bf16_input(200 + r, n) for r in order}
        m = Members(inputs, order)
        want = oracle.member_sum([bits(inputs[r]) for r in order])
        for r in order:
            words[r] = 1
        ext.local_reduce(m.bufs, flags_dev, m.order, m.out, 1, 3_000_000_000, 0, m.state)
        torch.cuda.synchronize()
        assert m.status() == (1, 0, 0)
        assert np.array_equal(bits(m.out), want)
        m.out.zero_()
        for r in order:
            words[r] = 0 if r == 0 else 2
        torch.cuda.synchronize()
        ctrl.words[BOUND] = 100_000
        ext.local_reduce(m.bufs, flags_dev, m.order, m.out, 2, 3_000_000_000, ctrl.dev, m.state)
        try:
            waited = named(ctrl, 1 << 0)
        finally:
            words[0] = 2
        torch.cuda.synchronize()
        assert waited, "the call never named row 0 as late: it did not wait for it"
        assert m.status() == (2, 0, 0)
        assert int(ctrl.words[LATE]) == 0
        assert np.array_equal(bits(m.out), want)
        assert not m.state[1:].any()
    finally:
        ctrl.close()
        ext.host_free(flags_host)


def test_a_late_member_that_never_comes_reads_as_zeros_mid_order(ext):
    """A member missing at the first read and never arriving: the members loaded before the wait
    are summed with zeros in its place, and the timeout names it."""
    n = 256 * 8192 + 13
    order = [2, 7, 4, 1]
    inputs = {r: bf16_input(80 + r, n) for r in order}
    m = Members(inputs, order)
    m.publish(epoch=5)
    m.publish(epoch=4, rows=[4])
    ext.local_reduce(m.bufs, m.flags, m.order, m.out, 5, 1_000_000, 0, m.state)  # 1 ms
    torch.cuda.synchronize()
    assert m.status() == (5, 2, 1 << 4)
    want, reason, late = oracle.reduce_protocol({r: bits(x) for r, x in inputs.items()},
                                                {r: (4 if r == 4 else 5) for r in order}, order, 5)
    assert (reason, late) == (2, 1 << 4)
    assert np.array_equal(bits(m.out), want)


@pytest.mark.parametrize("n", [2048, 8 * 256 * 4 * 3 + 6, 81920 + 6, 256 * 8192])
def test_a_captured_reduction_replays_like_eager_calls(ext, n):
    """The reduce records no memset and resets its own counters, so a HIP graph of it replays
    right: several replays, with eager work and synchronisations between them, each checked. One
    size per kernel: a grid of one (nothing counted), 12 workgroups (counted in the top word), 40
    workgroups and C5 (counted in two levels, at 1 and 4 vectors a thread)."""
    order = [3, 1, 2]
    inputs = {r: bf16_input(70 + r, n) for r in order}
    m = Members(inputs, order)
    m.publish(epoch=5)
    want = oracle.member_sum([bits(inputs[r]) for r in order])
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        ext.local_reduce(m.bufs, m.flags, m.order, m.out, 5, 10**9, 0, m.state)
    for i in range(4):
        m.out.fill_(i)  # eager work between the replays
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(bits(m.out), want), i
        assert m.status() == (5, 0, 0)
        assert not m.state[1:].any()


@pytest.mark.parametrize("n", [2048, 24576, 81920, 256 * 8192])
def test_an_order_naming_a_row_out_of_range_adds_nothing_and_says_so(ext, n):
    """Rows 9 and -1 in the order (outside [0, MAX_ROWS)) are not waited for and add nothing: the
    sum equals the valid members' ordered sum, bit for bit, and the outcome carries reason
    EVS_REDUCE_BAD_ORDER (4) through every counting mode: a grid of one, 12 workgroups (the top
    word), 40 (two levels) and C5."""
    inputs = {r: bf16_input(300 + r, n) for r in (0, 1)}
    m = Members(inputs, [1, 0])
    m.order.copy_(torch.tensor([4, 1, 9, 0, -1] + [0] * (MAXW - 4), dtype=torch.int32))
    m.publish(epoch=6)
    ext.local_reduce(m.bufs, m.flags, m.order, m.out, 6, 10**9, 0, m.state)
    torch.cuda.synchronize()
    assert m.status() == (6, 4, 0)
    assert np.array_equal(bits(m.out), oracle.member_sum([bits(inputs[1]), bits(inputs[0])]))
    assert not m.state[1:].any()


@pytest.mark.parametrize("order", [[0], [0, 1], [1, 0, 2], [0, 3], [3, 0], [2, 0, 1, 3]])
def test_special_values_round_as_the_oracle_does(ext, order):
    """Every bf16 pattern (signed zeros, subnormals, the largest values, infinities, NaNs), sums
    that overflow, inf meeting -inf, and exact ties: the kernel's fp32 adds keep subnormals and
    its rounding matches the oracle's bit for bit (tests/cases.py:special_members)."""
    members = special_members()
    inputs = {r: bf16_tensor(members[r]) for r in order}
    m = Members(inputs, order)
    m.publish(epoch=1)
    ext.local_reduce(m.bufs, m.flags, m.order, m.out, 1, 10**9, 0, m.state)
    torch.cuda.synchronize()
    assert np.array_equal(bits(m.out), oracle.member_sum([members[r] for r in order]))
    assert m.status() == (1, 0, 0)
