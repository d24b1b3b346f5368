"""Direct-transport calls at the sizes whose data meets in LDS, against the kernels whose data
meets in registers (which a tuning key of theirs asks for) over every form of buffers that a call
takes, and against the oracle: bit for bit, nothing written outside a buffer."""
import numpy as np
import pytest

import gpu_ipc_example_amd as vr
from gpu_ipc_example_amd.binding import DeviceBuffer
from tests.oracle_lib import BF16, DIST_NORMAL, F16

pytestmark = pytest.mark.gpu
SLACK = 256


def call(oracle, ctx, algo, ins, form, registers):
    """The bytes of every buffer after one call."""
    N, n = ctx.nranks, len(ins[0])
    src = [DeviceBuffer(n * 2 + SLACK) for _ in range(N)]
    dst = [DeviceBuffer(n * 2 + SLACK) for _ in range(N)] if form in ("apart", "apart by 8") else []
    for b in src + dst:
        b.fill(0xAB)
    at = [8 * (r % 3) if form == "apart by 8" else 8 if form == "in place at 8" else 0 for r in range(N)]
    for b, a, o in zip(src, ins, at):
        b.upload(a, o)
    bufs = [b.ptr + o for b, o in zip(src, at)]
    outs = None
    if dst:
        outs = [b.ptr + (40 + 8 * (r % 2) if form == "apart by 8" else 0) for r, b in enumerate(dst)]
    elif form == "each other's":
        outs = bufs[1:] + bufs[:1]
    elif form == "one for all":
        bufs, outs = bufs[:1] * N, None
    if registers:
        ctx.set_tuning(unroll=1)
    ctx.allreduce(algo, bufs, n, outs=outs, transport=vr.TRANSPORT_DIRECT)
    ctx.check()
    ctx.set_tuning(unroll=-1)
    got = [b.download(np.uint16, n + SLACK // 2) for b in src + dst]
    for b in src + dst:
        b.free()
    return got


@pytest.mark.parametrize("nranks,algo,mib", [(2, "simple", 62), (2, "small_ring", 66), (4, "bisect", 29), (4, "small_pcie", 97),
                                             (8, "small", 6), (8, "simple_ring", 14), (8, "bisect", 40), (8, "simple_transmit", 113),
                                             (8, "bisect", 98), (16, "bisect", 1), (16, "bisect", 30), (16, "bisect", 125)])
def test_same_as_through_registers(oracle, nranks, algo, mib):
    ctx = vr.VirtualRanks(nranks)
    msg = 16 if algo in ("small_ring", "simple_ring", "small_pcie") else 8
    n = ((mib << 20) // nranks ** 2 // 1024 * 1024 + 1000 + msg) // 16 * 16 // 2 * nranks
    if msg == 8:
        n += 4 * nranks
    for dtype, forms in ((F16, ("in place", "apart", "each other's", "one for all")), (BF16, ("in place", "apart by 8", "in place at 8"))):
        ctx.set_dtype(1 if dtype == BF16 else 0)
        ins = [oracle.generate_dt(dtype, n, 90_000 + r, DIST_NORMAL, 0.0, 1.0) for r in range(nranks)]
        for form in forms:
            if msg == 16 and form.endswith("8"):
                continue
            got = call(oracle, ctx, algo, ins, form, False)
            for k, (a, b) in enumerate(zip(got, call(oracle, ctx, algo, ins, form, True))):
                assert (a == b).all(), (form, k)
            if form == "in place":
                want = oracle.order_dt(dtype, 2 if algo == "bisect" else 1, ins)
                for r, g in enumerate(got):
                    assert oracle.count_mismatch_dt(dtype, g[:n], want) == 0, r
                    assert (g[n:] == 0xABAB).all(), r
    ctx.close()


@pytest.mark.parametrize("nranks,mib", [(2, 15), (2, 97), (4, 11), (4, 15), (8, 15)])
@pytest.mark.parametrize("form", ["apart", "own slot", "the next rank's slot"])
def test_gather_same_as_through_registers(oracle, nranks, mib, form):
    """Inputs of their own, and inputs that already are their slot of an output."""
    ctx = vr.VirtualRanks(nranks)
    n = ((mib << 20) // nranks // 16 * 16 + 48) // 2
    ins = [oracle.generate_dt(F16, n, 91_000 + r, DIST_NORMAL, 0.0, 1.0) for r in range(nranks)]
    want = oracle.allgather(ins)
    for registers in (False, True):
        outs = [DeviceBuffer(nranks * n * 2 + SLACK) for _ in range(nranks)]
        apart = [DeviceBuffer(n * 2 + SLACK) for _ in range(nranks)] if form == "apart" else []
        for b in outs:
            b.fill(0xAB)
        if apart:
            where = [(b, 16) for b in apart]
        else:
            where = [(outs[(q + (form != "own slot")) % nranks], q * n * 2) for q in range(nranks)]
        for (b, o), a in zip(where, ins):
            b.upload(a, o)
        if registers:
            ctx.set_tuning(unroll=1)
        ctx.allgather("allgather_simple", [b.ptr + o for b, o in where], [b.ptr for b in outs], n)
        ctx.check()
        ctx.set_tuning(unroll=-1)
        for r, b in enumerate(outs):
            got = b.download(np.uint16, nranks * n + SLACK // 2)
            assert (got[:nranks * n] == want).all() and (got[nranks * n:] == 0xABAB).all(), (registers, r)
        for b in outs + apart:
            b.free()
    ctx.close()
