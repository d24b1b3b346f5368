"""What a program that uses this library has it do, as timed cases.

Every case is one collective over N virtual ranks' device buffers through the
package's entry points, the way a caller's loop issues it: `VirtualRanks.allreduce`,
`.allgather` or `.allreduce_static`, buffers and context in hand, asynchronous on
the null stream.  The ranges that the listed cases stand for, and that `draw`
samples:

* sizes from 1 KiB per rank, where a call is one short launch, to 2 GiB of inputs
  (the size sweep's 8 x 256 MiB); any element count that the protocol's messages
  allow, so chunks that are odd multiples of 8 bytes are as common as even ones;
* 2, 4, 8 and 16 ranks as far as a protocol runs on them;
* binary16 and bfloat16;
* in place (the reference's semantics) and out of place;
* the default transport of every protocol, message passing on request, and the
  allocation-free entry point that callers under graph capture use.

Sums have a fixed association, so every result is exact to the bit.  An in-place
case works on its own results when it is called again, as a caller does who calls
twice: sums over equal ranks grow to infinities after some passes and stay there;
the time of a pass does not depend on the values.

Not here: launches that hold some of the ranks (`allreduce_rank`, `allreduce_ranks`).
They form a collective only with launches on other streams or in other processes,
and run the kernels of the message-passing cases below.
"""
import math

import torch

import gpu_ipc_example_amd as vr
from gpu_ipc_example_amd.binding import DTYPE_BF16, DTYPE_F16

KiB, MiB = 1 << 10, 1 << 20

# Protocols by sizeof(message_t) and the rank counts they run on.
ALGOS_8B = ("small", "simple", "bisect", "simple_transmit")
ALGOS_16B = ("small_pcie_p", "simple_pcie_p", "small_ring", "simple_ring", "small_pcie", "simple_pcie")
GATHERS = ("allgather_small", "allgather_simple")


def _case(name, algo, ranks, nelems, dtype="f16", transport="default", in_place=True, sigma=1.0):
    return {"name": name, "algo": algo, "ranks": ranks, "nelems": nelems, "dtype": dtype,
            "transport": transport, "in_place": in_place, "sigma": sigma}


def listed():
    return [
        # the smallest configured call, 2 ranks x 32 KiB: nothing but the call and one launch
        _case("simple_2x32KiB", "simple", 2, 16384),
        # the latency configuration: a decode step's activations, 1 MiB on each of 8 ranks
        _case("small_8x1MiB", "small", 8, 524288),
        # the bandwidth configuration: gradients of a layer, 32 MiB per rank, inputs kept
        _case("bisect_8x32MiB", "bisect", 8, 16777216, in_place=False, sigma=0.02),
        # the all-gather configuration: sharded weights, 8 MiB per rank
        _case("allgather_4x8MiB", "allgather_simple", 4, 4194304, in_place=False, sigma=1.0),
        # the size sweep's protocol (message passing by default): its smallest point,
        _case("parallel_8x4KiB", "parallel", 8, 2048),
        # the middle of its range, in the element type that the reference's program runs,
        _case("parallel_8x1MiB_bf16", "parallel", 8, 524288, dtype="bf16"),
        # and its largest point
        _case("parallel_8x256MiB", "parallel", 8, 134217728),
        # 16 ranks and a length that is no power of two: chunks of an odd number of 8-byte messages
        _case("bisect_16x12MB_bf16", "bisect", 16, 64 * 93751, dtype="bf16", in_place=False, sigma=0.02),
        # 4 ranks in place at an ordinary size with such a length
        _case("simple_4x20MB", "simple", 4, 16 * 625001),
        # neighbour-ring message passing on request, ragged length
        _case("ring_wire_4x8MB", "simple_ring", 4, 32 * 125003, transport="wire", in_place=False),
        # message-passing all-gather on request, ragged length
        _case("allgather_wire_8x1MB", "allgather_simple", 8, 8 * 65537, transport="wire", in_place=False),
        # the allocation-free call that a captured decode step makes
        _case("static_8x256KiB", "small", 8, 131072, transport="static"),
    ]


def _length(rng, unit, most_bytes):
    """An element count per rank, log-uniform from 1 KiB to most_bytes, in whole messages."""
    nbytes = math.exp(rng.uniform(math.log(KiB), math.log(most_bytes)))
    return max(1, int(nbytes / 2 / unit)) * unit


def draw(rng):
    dtype = "bf16" if rng.random() < 0.3 else "f16"
    in_place = rng.random() < 0.5
    kind = rng.choice(["allreduce"] * 5 + ["parallel"] * 2 + ["wire"] * 2 + ["gather"] * 2 + ["static"])
    transport, most = "default", 2048 * MiB            # most: bytes of all ranks' inputs
    if kind == "gather":
        algo, ranks = rng.choice(GATHERS), rng.choice((2, 4, 8))
        if rng.random() < 0.3:
            transport, most = "wire", 512 * MiB // ranks
        else:
            most = 2048 * MiB // ranks
        n, in_place = _length(rng, 8, most // ranks), False
    else:
        if kind == "parallel":
            algo = "parallel"
        elif kind == "static":
            algo = rng.choice([a for a in ALGOS_8B + ALGOS_16B if a != "simple_transmit"])
            transport, most = "static", 64 * MiB
        else:
            algo = rng.choice(ALGOS_8B[:3] * 2 + ALGOS_8B[3:] + ALGOS_16B)
            if kind == "wire":
                transport, most = "wire", 512 * MiB
        ranks = rng.choice((2, 4, 8))
        if algo == "bisect":
            ranks = rng.choice((4, 8) if transport == "static" else (4, 8, 16))
        n = _length(rng, (8 if algo in ALGOS_16B else 4) * ranks, min(most // ranks, 256 * MiB))
    c = _case("", algo, ranks, n, dtype, transport, in_place, rng.choice((0.02, 1.0)))
    del c["name"]
    return c


def prepare(case, seed):
    n, ne = case["ranks"], case["nelems"]
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float16
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ins = []
    for _ in range(n):
        x = torch.empty(ne, dtype=dtype, device="cuda")
        ins.append(x.normal_(0.0, case["sigma"], generator=gen))
    gather = case["algo"].startswith("allgather")
    outs = ins
    if gather:
        outs = [torch.empty(n * ne, dtype=dtype, device="cuda") for _ in range(n)]
    elif not case["in_place"]:
        outs = [torch.empty(ne, dtype=dtype, device="cuda") for _ in range(n)]
    ctx = vr.VirtualRanks(n)
    ctx.set_dtype(DTYPE_BF16 if case["dtype"] == "bf16" else DTYPE_F16)
    if case["transport"] == "wire" or (case["transport"] == "default" and case["algo"] == "parallel"):
        ctx.reserve_wire()
    return {"ctx": ctx, "case": case, "gather": gather, "ins": ins, "outs": outs}


def run(state):
    case, ctx, outs = state["case"], state["ctx"], state["outs"]
    src = [t.data_ptr() for t in state["ins"]]
    dst = None if outs is state["ins"] else [t.data_ptr() for t in outs]
    transport = vr.TRANSPORT_WIRE if case["transport"] == "wire" else vr.TRANSPORT_DEFAULT
    if state["gather"]:
        ctx.allgather(case["algo"], src, dst, case["nelems"], transport=transport)
    elif case["transport"] == "static":
        ctx.allreduce_static(case["algo"], src, case["nelems"], outs=dst)
    else:
        ctx.allreduce(case["algo"], src, case["nelems"], outs=dst, transport=transport)
    return outs


def work(case):
    n, ne = case["ranks"], case["nelems"]
    if case["algo"].startswith("allgather"):
        return {"bytes": 2 * ne * n * (1 + n), "flops": 0}      # every slice read once, written to every rank
    return {"bytes": 2 * ne * n * 2, "flops": (n - 1) * ne}     # every input read once, every output written once


def tolerance(case):
    return "exact"
