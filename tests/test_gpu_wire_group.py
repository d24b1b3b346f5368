"""Wire-transport launches that hold all ranks (messages through LDS) at the sizes where
the work-group form can go wrong, bit for bit against the oracle.  A wave's wire is 1 KiB
of a chunk, 2 or 4 KiB where a lane carries two or four vectors (as the sizes of inputs given
below make it); a chunk of 8-byte messages may end inside a lane's 16 bytes."""
import numpy as np
import pytest

import gpu_ipc_example_amd as vr
from gpu_ipc_example_amd.binding import DeviceBuffer
from tests.oracle_lib import BF16, DIST_NORMAL, F16
from tests.test_gpu_wire import run_allgather_wire

pytestmark = pytest.mark.gpu
WIRE = vr.TRANSPORT_WIRE


def run(oracle, ctx, algo, n, dtype, inplace, offset, seed):
    N = ctx.nranks
    ctx.set_dtype(1 if dtype == BF16 else 0)
    ins = [oracle.generate_dt(dtype, n, seed + r, DIST_NORMAL, 0.0, 1.0) for r in range(N)]
    want = oracle.order_dt(dtype, 2 if algo == "bisect" else 1, ins)
    what = (algo, N, n, dtype, inplace, offset)
    src = [DeviceBuffer(n * 2 + 64) for _ in range(N)]
    dst = src if inplace else [DeviceBuffer(n * 2 + 64) for _ in range(N)]
    for b in src + dst:
        b.fill(0xAB)
    for b, a in zip(src, ins):
        b.upload(a, offset)
    ctx.allreduce(algo, [b.ptr + offset for b in src], n,
                  outs=None if inplace else [b.ptr + offset for b in dst], transport=WIRE)
    ctx.check()
    for r, b in enumerate(dst):
        got = b.download(np.uint16, n + 32)
        assert oracle.count_mismatch_dt(dtype, got[offset // 2:offset // 2 + n], want) == 0, (what, r)
        # nothing is written around the buffer
        assert (got[:offset // 2] == 0xABAB).all() and (got[offset // 2 + n:] == 0xABAB).all(), (what, r)
    for b in src + (dst if dst is not src else []):
        b.free()


@pytest.mark.parametrize("nranks,algo", [(2, "simple"), (4, "parallel"), (8, "parallel"), (8, "simple_transmit"),
                                         (4, "bisect"), (8, "bisect"), (16, "bisect"), (2, "simple_ring"),
                                         (8, "simple_ring"), (8, "simple_pcie")])
def test_edges_of_a_wire(oracle, nranks, algo):
    msg = 16 if algo in ("simple_ring", "simple_pcie") else 8
    ctx = vr.VirtualRanks(nranks)
    for k, chunk in enumerate((msg, 1024 - msg, 1024, 1024 + msg, 2048 - msg, 2048, 2048 + msg, 5 * 2048 + 3 * msg)):
        for dtype in (F16, BF16):
            for inplace in (True, False):
                for offset in (0, 8) if msg == 8 else (0,):
                    run(oracle, ctx, algo, nranks * chunk // 2, dtype, inplace, offset, 40_000 + 100 * k)
    ctx.close()


@pytest.mark.parametrize("algo,mib", [("simple_ring", 34), ("simple_pcie", 34), ("bisect", 20), ("parallel", 66),
                                      ("parallel", 514)])
def test_ragged_sizes_of_the_larger_launches(oracle, algo, mib):
    """Eight ranks, just inside the sizes that change the vectors per lane, the residency and
    (in place) the cache policy."""
    ctx = vr.VirtualRanks(8)
    msg = 16 if algo in ("simple_ring", "simple_pcie") else 8
    chunk = (mib << 20) // 64 + 3 * msg
    run(oracle, ctx, algo, 8 * chunk // 2, F16, True, 0, 50_000)
    ctx.close()


@pytest.mark.parametrize("nranks,algo,kib", [(2, "simple", 12 * 1024), (4, "bisect", 12 * 1024), (8, "parallel", 8 * 1024),
                                             (8, "small_pcie", 14 * 1024), (8, "bisect", 80 * 1024),
                                             (8, "simple_transmit", 20 * 1024), (16, "bisect", 30 * 1024),
                                             (8, "simple_ring", 14 * 1024), (8, "small_ring", 110 * 1024)])
def test_vectors_per_lane(oracle, nranks, algo, kib):
    """One, two and four vectors per lane: messages of 1, 2 and 4 KiB whose last ends early, and a wave's
    share of the sums in each width; rings by columns and by chunks."""
    msg = 16 if algo.endswith(("pcie", "ring")) else 8
    ctx = vr.VirtualRanks(nranks)
    chunk = kib * 1024 // nranks ** 2 // 4096 * 4096
    for k, tail in enumerate((0, msg, 1024 - msg, 3072 + msg)):
        run(oracle, ctx, algo, nranks * (chunk + tail) // 2, BF16 if k % 2 else F16, k < 2, 0, 46_000 + 100 * k)
    ctx.close()


@pytest.mark.parametrize("nranks", [2, 8])
def test_allgather_edges(oracle, nranks):
    ctx = vr.VirtualRanks(nranks)
    for n in (8, 504, 512, 520, 8 * 643):
        ins = [oracle.generate_dt(F16, n, 60_000 + r, DIST_NORMAL, 0.0, 1.0) for r in range(nranks)]
        want = oracle.allgather(ins)
        for alias in (False, True):
            for r, got in enumerate(run_allgather_wire(ctx, "allgather_simple", ins, alias)):
                assert (got == want).all(), (n, r, alias)
    ctx.close()


@pytest.mark.parametrize("nranks,algo,mib,inplace", [(4, "simple_ring", 194, True), (4, "bisect", 194, False),
                                                     (8, "simple", 71, True), (16, "bisect", 98, False)])
def test_capped_and_resident_launches(oracle, nranks, algo, mib, inplace):
    """Just inside the sizes (bytes of all ranks' inputs) that cap the work-groups per compute unit,
    the largest that stay cacheable in place, and sixteen ranks with one vector per lane, with a
    chunk that ends inside a wire."""
    ctx = vr.VirtualRanks(nranks)
    msg = 16 if algo == "simple_ring" else 8
    chunk = (mib << 20) // nranks ** 2 // 16 * 16 + 3 * msg
    run(oracle, ctx, algo, nranks * chunk // 2, F16, inplace, 0, 70_000)
    ctx.close()


@pytest.mark.parametrize("nranks,kib", [(8, 512), (8, 1024), (4, 700), (4, 3 * 1024), (2, 6 * 1024), (2, 12 * 1024),
                                        (8, 10 * 1024)])
def test_runs_of_a_gather(oracle, nranks, kib):
    """KiB of input per rank at which work-groups are permuted (in runs of 16 and 64 KiB, with one,
    two and four vectors per lane) and at which they are not: a last group that is whole, and ragged ones."""
    ctx = vr.VirtualRanks(nranks)
    for tail in (0, 16, 9 * 1024 + 1008):
        n = (kib * 1024 + tail) // 2
        ins = [oracle.generate_dt(F16, n, 72_000 + r, DIST_NORMAL, 0.0, 1.0) for r in range(nranks)]
        want = oracle.allgather(ins)
        for r, got in enumerate(run_allgather_wire(ctx, "allgather_simple", ins, tail == 16)):
            assert (got == want).all(), (n, r)
    ctx.close()


def test_allgather_beyond_half_the_cache(oracle):
    """Four ranks with 4 x 33 MiB of inputs and a ragged slice: capped, results streamed past cached inputs."""
    ctx = vr.VirtualRanks(4)
    n = (33 << 19) + 24
    ins = [oracle.generate_dt(F16, n, 71_000 + r, DIST_NORMAL, 0.0, 1.0) for r in range(4)]
    want = oracle.allgather(ins)
    for r, got in enumerate(run_allgather_wire(ctx, "allgather_simple", ins, False)):
        assert (got == want).all(), r
    ctx.close()


@pytest.mark.parametrize("nranks,algo", [(2, "simple"), (8, "parallel"), (4, "bisect"), (16, "bisect"), (8, "simple_transmit"),
                                         (8, "simple_ring"), (8, "simple_pcie")])
def test_chunks_of_several_launches(oracle, nranks, algo):
    """Chunks longer than one launch covers: whole and ragged last segments, starts of segments
    inside a vector (offset 8) and inside a line."""
    msg = 16 if algo in ("simple_ring", "simple_pcie") else 8
    ctx = vr.VirtualRanks(nranks)
    for kib in (1, 3):
        ctx.set_tuning(segment_kib=kib)
        for k, chunk in enumerate((1024 * kib - msg, 1024 * kib, 1024 * kib + msg, 4 * 1024 * kib, 4 * 1024 * kib + 5 * msg)):
            for inplace in (True, False):
                for offset in (0, 8) if msg == 8 else (0, 16):
                    run(oracle, ctx, algo, nranks * chunk // 2, F16, inplace, offset, 80_000 + 100 * k)
    ctx.close()


def test_gathers_of_several_launches(oracle):
    ctx = vr.VirtualRanks(8)
    ctx.set_tuning(segment_kib=1)
    for n in (504, 512, 520, 8 * 643):
        ins = [oracle.generate_dt(F16, n, 81_000 + r, DIST_NORMAL, 0.0, 1.0) for r in range(8)]
        want = oracle.allgather(ins)
        for alias in (False, True):
            for r, got in enumerate(run_allgather_wire(ctx, "allgather_simple", ins, alias)):
                assert (got == want).all(), (n, r, alias)
    ctx.close()
