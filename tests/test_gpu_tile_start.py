"""Tiles laid on KiBs (direct) and 128-byte lines of the outputs: buffers that start anywhere on 8 bytes, chunks
that are any multiple of 8 bytes, buffers that disagree about their place in 16 bytes.  Bit for
bit against the oracle, nothing written outside a buffer, inputs kept."""
import numpy as np
import pytest

import gpu_ipc_example_amd as vr
from gpu_ipc_example_amd.binding import DeviceBuffer
from tests import vr_helpers as H

pytestmark = pytest.mark.gpu


def run(oracle, ctx, algo, n, offsets, out_offsets, transport, seed, slack=256):
    N = ctx.nranks
    ins = H.make_inputs(oracle, N, n, seed)
    want = H.expected(oracle, algo, ins)
    what = (algo, N, n, offsets, out_offsets, transport)
    src = [DeviceBuffer(n * 2 + slack) for _ in range(N)]
    dst = [DeviceBuffer(n * 2 + slack) for _ in range(N)] if out_offsets else src
    for b in src + dst:
        b.fill(0xAB)
    for b, a, o in zip(src, ins, offsets):
        b.upload(a, o)
    outs = [b.ptr + o for b, o in zip(dst, out_offsets)] if out_offsets else None
    ctx.allreduce(algo, [b.ptr + o for b, o in zip(src, offsets)], n, outs=outs, transport=transport)
    ctx.check()
    for r, (b, o) in enumerate(zip(dst, out_offsets or offsets)):
        got = b.download(np.uint16, n + slack // 2)
        assert oracle.count_mismatch(got[o // 2:o // 2 + n], want) == 0, (what, r)
        assert (got[:o // 2] == 0xABAB).all() and (got[o // 2 + n:] == 0xABAB).all(), (what, r)
    if out_offsets:
        for b, o, a in zip(src, offsets, ins):
            assert (b.download(np.uint16, n, o) == a).all(), what
    for b in src + (dst if dst is not src else []):
        b.free()


@pytest.mark.parametrize("nranks,algo", [(2, "simple"), (4, "bisect"), (8, "small"), (8, "bisect"), (16, "bisect")])
def test_direct(oracle, nranks, algo):
    ctx = vr.VirtualRanks(nranks)
    knobs = (dict(), dict(oneshot=1, block=64, unroll=1, deal=1), dict(oneshot=0, block=64, unroll=2, waves_per_cu=1),
             dict(oneshot=1, block=64, unroll=4, segment_kib=1))
    for k, kn in enumerate(knobs):
        ctx.set_tuning(**kn)
        for chunk in (8, 120, 1016, 1032, 2048, 9 * 1024 + 24):
            n = nranks * chunk // 2
            for off in (0, 8, 16, 120):
                run(oracle, ctx, algo, n, [off] * nranks, None, vr.TRANSPORT_DIRECT, 70_000 + chunk)
            run(oracle, ctx, algo, n, [24] * nranks, [88] * nranks, vr.TRANSPORT_DIRECT, 71_000 + chunk)
            run(oracle, ctx, algo, n, [8 * (r % 3) for r in range(nranks)], [8 + 16 * (r % 2) for r in range(nranks)],
                vr.TRANSPORT_DIRECT, 72_000 + chunk)
        ctx.set_tuning(**{key: -1 for key in kn})
    ctx.close()


@pytest.mark.parametrize("transport", [vr.TRANSPORT_DIRECT, vr.TRANSPORT_WIRE])
@pytest.mark.parametrize("nranks,algo", [(2, "simple"), (8, "parallel"), (16, "bisect")])
def test_places_within_a_kib(oracle, nranks, algo, transport):
    """First tiles that hold 16 bytes of the chunk, or all but 16."""
    ctx = vr.VirtualRanks(nranks)
    for chunk in (8, 1024, 3 * 1024 + 520):
        for off in (264, 1008, 1016):
            n = nranks * chunk // 2
            run(oracle, ctx, algo, n, [off] * nranks, None, transport, 76_000 + chunk, 2048)
            run(oracle, ctx, algo, n, [8] * nranks, [off] * nranks, transport, 77_000 + chunk, 2048)
    ctx.close()


@pytest.mark.parametrize("nranks,algo", [(4, "parallel"), (8, "parallel"), (8, "simple_transmit"), (16, "bisect")])
def test_wire(oracle, nranks, algo):
    ctx = vr.VirtualRanks(nranks)
    for chunk in (8, 1016, 2056, 9 * 1024 + 24):
        n = nranks * chunk // 2
        for off in (0, 8, 120):
            run(oracle, ctx, algo, n, [off] * nranks, None, vr.TRANSPORT_WIRE, 73_000 + chunk)
        run(oracle, ctx, algo, n, [8 * (r % 3) for r in range(nranks)], [40 + 8 * (r % 2) for r in range(nranks)],
            vr.TRANSPORT_WIRE, 74_000 + chunk)
    ctx.close()


@pytest.mark.parametrize("transport", [vr.TRANSPORT_DIRECT, vr.TRANSPORT_WIRE])
def test_allgather(oracle, transport):
    """Slices of any multiple of 16 bytes behind outputs at any multiple of 16."""
    ctx = vr.VirtualRanks(8)
    for n in (8, 504, 520, 8 * 1027):
        ins = [oracle.generate(n, 75_000 + r, 1, 0.0, 1.0) for r in range(8)]
        want = oracle.allgather(ins)
        for o in (0, 48, 112):
            src = [DeviceBuffer(n * 2 + 256) for _ in range(8)]
            dst = [DeviceBuffer(8 * n * 2 + 256) for _ in range(8)]
            for b, a in zip(src, ins):
                b.upload(a, 16)
            for b in dst:
                b.fill(0xAB)
            ctx.allgather("allgather_simple", [b.ptr + 16 for b in src], [b.ptr + o for b in dst], n, transport=transport)
            ctx.check()
            for r, b in enumerate(dst):
                got = b.download(np.uint16, 8 * n + 128)
                assert (got[o // 2:o // 2 + 8 * n] == want).all(), (n, o, r)
                assert (got[:o // 2] == 0xABAB).all() and (got[o // 2 + 8 * n:] == 0xABAB).all(), (n, o, r)
            for b in src + dst:
                b.free()
    ctx.close()
