"""The copies a program makes through this library, as measurable cases.

Each case is a dict of plain values.  ``prepare`` builds what the program
holds before the call (device buffers, committed types, batches), ``run``
makes one pass through the public entry points, and ``work`` counts the bytes
the pass cannot avoid moving: every packed byte is read once and written once,
by the pack and again by the unpack.  All outputs are bytes: packed streams,
and whole destination buffers, gaps between the type's blocks included.

Kinds:

* ``mpi``       MPI_Pack then MPI_Unpack of one derived type, each returning
                when its copy is done; the packed side in device memory or in
                mapped host memory (the one-shot target).
* ``stream``    the same copies enqueued on the library stream without
                waiting (tempi_pack_sb, tempi_unpack_sb).
* ``faces``     the three low faces of one grid, packed by one batch launch
                and unpacked into a second grid's ghost cells by another.
* ``halo``      the 26 halo regions of many subdomains, the same two batches.
* ``random``    a batch of unrelated 1D, 2D and 3D requests, packed.
* ``sendrecv``  MPI_Irecv, MPI_Isend and MPI_Waitall of a derived type in
                device memory, to the process itself.
* ``neighbor``  one MPI_Neighbor_alltoallw halo exchange of a periodic
                subdomain whose 26 neighbours are the process itself.
"""
import ctypes
import itertools
import math
import random

import numpy as np
import torch

import tempi_amd as ta
from tempi_amd import mpi as tmpi

BYTE = ("named", "MPI_BYTE")
BLOCKS = (1, 3, 4, 8, 12, 16, 24, 32, 64, 100, 128, 256, 512, 1024)


def listed():
    return [
        # one small message: 16 blocks of 64 B, all launch and completion
        _mpi("mpi_1k", rows=16, block=64, stride=512),
        # a plain 2D type of ordinary size, vector(1024, 256, 512)
        _mpi("mpi_256k", rows=1024, block=256, stride=512),
        # two objects of 4 MiB in 32-B blocks 512 B apart, the largest type of
        # the 2D MPI_Pack sweep
        _mpi("mpi_2x4m", rows=131072, block=32, stride=512, count=2),
        # the one-shot send's pack: 4 MiB of 64-B blocks into host memory
        _mpi("mapped_4m", rows=65536, block=64, stride=512, mapped=True),
        # rows of three floats at an odd stride from an odd address, 3D
        _stream("stream_12b", planes=5, rows=131072, block=12, stride=1001, pad=37, base=5),
        # 64-B rows that start anywhere in a line
        _stream("stream_64b_odd", planes=1, rows=524288, block=64, stride=1777, pad=0, base=5),
        # a large aligned copy, 256 MiB of 64-B rows
        _stream("stream_64b_256m", planes=1, rows=4194304, block=64, stride=192, pad=0, base=0),
        # the faces of a 512^3 float grid with three ghost cells
        {"name": "faces_518", "kind": "faces", "n": 512, "ghost": 3, "cell": 4},
        # the halo regions of 64 subdomains of 128^3 doubles, radius 3
        {"name": "halo_64", "kind": "halo", "subs": 64, "n": 128, "radius": 3, "cell": 8},
        # 4096 mixed requests of 64 B to 16 MiB
        {"name": "random_4096", "kind": "random", "requests": 4096, "most": 16 << 20, "mix": 4},
        # a small non-blocking exchange of device data
        {"name": "sendrecv_256k", "kind": "sendrecv", "rows": 1024, "block": 256, "stride": 512},
        # the halo exchange of one 128^3 double subdomain as one collective
        {"name": "neighbor_128", "kind": "neighbor", "n": 128, "radius": 3, "cell": 8},
    ]


def draw(rng):
    kind = rng.choice(("mpi", "mpi", "stream", "stream", "faces", "halo", "random", "sendrecv",
                       "neighbor"))
    if kind == "mpi":
        block = rng.choice(BLOCKS[:-1])
        mapped = rng.random() < 0.25
        rows = max(2, _log(rng, 1 << 10, 4 << 20) // block)
        return _mpi(None, rows=rows, block=block, stride=_gap(rng, block, 512),
                    count=rng.choice((1, 1, 2)), base=_base(rng), mapped=mapped)
    if kind == "stream":
        block = rng.choice(BLOCKS)
        planes = rng.choice((1, rng.randint(2, 8)))
        stride = _gap(rng, block, 4096)
        # at most 256 MiB packed and 4 GiB spanned
        most = min((256 << 20) // block, (4 << 30) // stride) // planes
        rows = _log(rng, max(2, (64 << 10) // (block * planes)), most)
        return _stream(None, planes=planes, rows=rows, block=block, stride=stride,
                       pad=rng.randint(0, 4096), base=_base(rng))
    if kind == "faces":
        return {"kind": kind, "n": _log(rng, 48, 512), "ghost": rng.randint(1, 4),
                "cell": rng.choice((4, 8))}
    if kind == "halo":
        return {"kind": kind, "subs": _log(rng, 1, 64), "n": _log(rng, 24, 128),
                "radius": rng.randint(1, 3), "cell": rng.choice((4, 8))}
    if kind == "random":
        return {"kind": kind, "requests": _log(rng, 16, 2048), "most": _log(rng, 1 << 14, 16 << 20),
                "mix": rng.randint(5, 1 << 20)}
    if kind == "sendrecv":
        block = rng.choice(BLOCKS[2:-1])
        return {"kind": kind, "rows": max(2, _log(rng, 1 << 10, 4 << 20) // block), "block": block,
                "stride": _gap(rng, block, 512)}
    return {"kind": kind, "n": _log(rng, 24, 128), "radius": rng.randint(1, 3),
            "cell": rng.choice((4, 8))}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    torch.cuda.synchronize()  # the library's stream does not wait for torch's
    return state


def run(state):
    return state["run"](state)


def work(case):
    # a pass that packs and unpacks moves every packed byte four times
    times = 2 if case["kind"] == "random" else 4
    return {"bytes": times * _PACKED[case["kind"]](case), "flops": 0}


# -- cases --------------------------------------------------------------------


def _mpi(name, rows, block, stride, count=1, base=0, mapped=False):
    c = {"kind": "mpi", "rows": rows, "block": block, "stride": stride, "count": count,
         "base": base, "mapped": mapped}
    return dict(c, name=name) if name else c


def _stream(name, planes, rows, block, stride, pad, base):
    c = {"kind": "stream", "planes": planes, "rows": rows, "block": block, "stride": stride,
         "pad": pad, "base": base}
    return dict(c, name=name) if name else c


def _log(rng, low, high):
    """An integer in [low, high], spread over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _gap(rng, block, most):
    """A stride: mostly any, sometimes one that keeps rows aligned."""
    gap = rng.randint(1, most)
    return block + gap if rng.random() < 0.6 else -(-(block + gap) // 64) * 64


def _base(rng):
    return rng.choice((0, 0, rng.randint(1, 15)))


# -- buffers and types ----------------------------------------------------------


def _random_bytes(n, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    words = torch.randint(-(1 << 63), (1 << 63) - 1, (-(-n // 8),), dtype=torch.int64,
                          device="cuda", generator=g)
    return words.view(torch.uint8)[:n]


def _filled(n):
    return torch.full((n,), 0xAB, dtype=torch.uint8, device="cuda")


def _normal_grid(cells, cell, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind = torch.float32 if cell == 4 else torch.float64
    return torch.randn(cells, dtype=kind, device="cuda", generator=g).view(torch.uint8)


def _vector(case):
    return ("vector", case["rows"], case["block"], case["stride"], BYTE)


def _commit(spec):
    m = tmpi.get()
    h = m.type_from_spec(spec)
    sb, size = m.strided_block(h)
    return h, sb, size


def _strided_block(spec):
    """What tempi_pack_sb and a batch take: the type itself is not kept."""
    h, sb, size = _commit(spec)
    tmpi.get().free(h)
    return sb, size


# -- MPI_Pack and MPI_Unpack ------------------------------------------------------


def _mpi_packed(case):
    return case["rows"] * case["block"] * case["count"]


def _mpi_prepare(case, seed):
    h, sb, size = _commit(_vector(case))
    span = case["base"] + sb.extent * case["count"]
    total = size * case["count"]
    state = {"run": _mpi_run, "mpi": tmpi.get(), "type": h, "count": case["count"],
             "src": _random_bytes(span, seed), "dst": _filled(span), "total": total}
    if case["mapped"]:
        buf = ta.DeviceBuffer(total, mapped=True)
        raw = (ctypes.c_uint8 * total).from_address(buf.addr())
        raw.owner = buf  # the memory lives as long as an array on it
        state.update(packed=np.frombuffer(raw, np.uint8), packed_at=buf.addr())
    else:
        state["packed"] = torch.empty(total, dtype=torch.uint8, device="cuda")
        state["packed_at"] = state["packed"].data_ptr()
    state["from"] = state["src"].data_ptr() + case["base"]
    state["to"] = state["dst"].data_ptr() + case["base"]
    return state


def _mpi_run(s):
    m = s["mpi"]
    err, _ = m.pack(s["from"], s["count"], s["type"], s["packed_at"], s["total"])
    err2, _ = m.unpack(s["packed_at"], s["total"], s["to"], s["count"], s["type"])
    if err or err2:
        raise RuntimeError(f"MPI_Pack {err}, MPI_Unpack {err2}")
    return s["packed"], s["dst"]


# -- the same copies on the library stream ------------------------------------------


def _stream_packed(case):
    return case["planes"] * case["rows"] * case["block"]


def _stream_prepare(case, seed):
    spec = _vector(case)
    if case["planes"] > 1:
        spec = ("hvector", case["planes"], 1, case["rows"] * case["stride"] + case["pad"], spec)
    sb, size = _strided_block(spec)
    span = case["base"] + sb.extent
    state = {"run": _stream_run, "sb": sb, "size": size, "src": _random_bytes(span, seed),
             "dst": _filled(span),
             "packed": torch.empty(size, dtype=torch.uint8, device="cuda")}
    state["from"] = state["src"].data_ptr() + case["base"]
    state["to"] = state["dst"].data_ptr() + case["base"]
    return state


def _stream_run(s):
    at = s["packed"].data_ptr()
    ta.pack_sb(s["sb"], s["from"], 1, at, s["size"])
    ta.unpack_sb(s["sb"], at, s["size"], s["to"], 1)
    return s["packed"], s["dst"]


# -- grid faces --------------------------------------------------------------------


def _face_specs(case, ghost):
    """The low faces of the grid's interior, or the ghost cells outside them."""
    n, g = case["n"], case["ghost"]
    cell = ("named", "MPI_FLOAT" if case["cell"] == 4 else "MPI_DOUBLE")
    for axis in (2, 1, 0):
        sub = [g if d == axis else n for d in range(3)]
        start = [0 if ghost and d == axis else g for d in range(3)]
        yield ("subarray", [n + 2 * g] * 3, sub, start, "C", cell)


def _faces_packed(case):
    return 3 * case["n"] ** 2 * case["ghost"] * case["cell"]


def _faces_prepare(case, seed):
    cells = (case["n"] + 2 * case["ghost"]) ** 3
    src = _normal_grid(cells, case["cell"], seed)
    dst = _filled(cells * case["cell"])
    packed = torch.empty(_faces_packed(case), dtype=torch.uint8, device="cuda")
    return _pack_unpack_batches([(0, s) for s in _face_specs(case, False)],
                                [(0, s) for s in _face_specs(case, True)], src, dst, packed)


def _pack_unpack_batches(send, recv, src, dst, packed):
    """Batches of (offset of the buffer, type) regions: out of src into
    packed, and from packed into dst."""
    blocks = {}

    def requests(regions, buf, direction):
        at = packed.data_ptr()
        for offset, spec in regions:
            key = repr(spec)
            if key not in blocks:
                blocks[key] = _strided_block(spec)
            sb, size = blocks[key]
            yield sb, buf.data_ptr() + offset, at, 1, direction
            at += size

    return {"run": _batches_run, "src": src, "dst": dst, "packed": packed,
            "pack": ta.Batch(requests(send, src, ta.DIR_PACK)),
            "unpack": ta.Batch(requests(recv, dst, ta.DIR_UNPACK))}


def _batches_run(s):
    s["pack"].launch()
    s["unpack"].launch()
    return s["packed"], s["dst"]


# -- halo regions of many subdomains ------------------------------------------------

DIRECTIONS = [d for d in itertools.product((-1, 0, 1), repeat=3) if d != (0, 0, 0)]


def _halo_region(case, direction, ghost):
    """The region of a subdomain that goes to `direction` (z, y, x), or the
    ghost cells that come from there."""
    n, r = case["n"], case["radius"]
    low = {-1: 0 if ghost else r, 0: r, 1: n + (r if ghost else 0)}
    sizes = [n + 2 * r] * 3
    subsizes = [n if d == 0 else r for d in direction]
    starts = [low[d] for d in direction]
    sizes[2], subsizes[2], starts[2] = (v[2] * case["cell"] for v in (sizes, subsizes, starts))
    return ("subarray", sizes, subsizes, starts, "C", BYTE)


def _halo_bytes(case):
    """Packed bytes of one subdomain's 26 regions."""
    n, r = case["n"], case["radius"]
    return ((n + 2 * r) ** 3 - n ** 3) * case["cell"]


def _halo_packed(case):
    return case["subs"] * _halo_bytes(case)


def _halo_prepare(case, seed):
    sub = (case["n"] + 2 * case["radius"]) ** 3 * case["cell"]
    # each subdomain starts at a multiple of 256 B, as an allocation does
    pitch = -(-sub // 256) * 256
    src = _random_bytes(case["subs"] * pitch, seed)
    dst = _filled(case["subs"] * pitch)
    packed = torch.empty(_halo_packed(case), dtype=torch.uint8, device="cuda")
    send = [(i * pitch, _halo_region(case, d, False))
            for i in range(case["subs"]) for d in DIRECTIONS]
    recv = [(i * pitch, _halo_region(case, tuple(-x for x in d), True))
            for i in range(case["subs"]) for d in DIRECTIONS]
    return _pack_unpack_batches(send, recv, src, dst, packed)


# -- unrelated requests ------------------------------------------------------------


def _random_blocks(case):
    """Strided blocks (start, extent, counts, strides) with packed sizes spread
    over the logarithm of 64 B to `most`, and the source bytes they reach."""
    rng = random.Random(case["mix"])
    out, reach = [], 0
    for _ in range(case["requests"]):
        target = int(math.exp(rng.uniform(math.log(64), math.log(case["most"]))))
        dims = rng.choice((1, 2, 3))
        counts, strides = [target], [1]
        if dims > 1:
            block = min(rng.choice((4, 8, 12, 16, 32, 64, 128, 256, 512, 1024, 2048)), target)
            rows = max(1, target // block)
            inner = rows if dims == 2 else max(1, math.isqrt(rows))
            stride = block + rng.randint(0, 512)
            counts, strides = [block, inner], [1, stride]
            if dims == 3:
                counts.append(max(1, rows // inner))
                strides.append(stride * inner + rng.randint(0, 4096))
        span = counts[0] + sum((c - 1) * s for c, s in zip(counts[1:], strides[1:]))
        start = 4 * rng.randint(0, 3)
        out.append((start, span + 16, counts, strides))
        reach = max(reach, start + span)
    return out, reach


def _random_packed(case):
    return sum(math.prod(counts) for _, _, counts, _ in _random_blocks(case)[0])


def _random_prepare(case, seed):
    blocks, reach = _random_blocks(case)
    src = _random_bytes(reach, seed)
    packed = torch.empty(_random_packed(case), dtype=torch.uint8, device="cuda")
    requests, at = [], packed.data_ptr()
    for b in blocks:
        sb = ta.StridedBlock.make(*b)
        requests.append((sb, src.data_ptr(), at, 1, ta.DIR_PACK))
        at += sb.size()
    return {"run": _random_run, "src": src, "packed": packed, "pack": ta.Batch(requests)}


def _random_run(s):
    s["pack"].launch()
    return s["packed"]


# -- point to point and neighbourhood exchanges ----------------------------------------


def _sendrecv_packed(case):
    return case["rows"] * case["block"]


def _sendrecv_prepare(case, seed):
    h, sb, _ = _commit(_vector(case))
    return {"run": _sendrecv_run, "mpi": tmpi.get(), "type": h,
            "src": _random_bytes(sb.extent, seed), "dst": _filled(sb.extent)}


def _sendrecv_run(s):
    m = s["mpi"]
    err, r = m.irecv(s["dst"].data_ptr(), 1, s["type"], 0, 41)
    err2, q = m.isend(s["src"].data_ptr(), 1, s["type"], 0, 41)
    err3, _, _ = m.waitall([r, q])
    if err or err2 or err3:
        raise RuntimeError(f"MPI_Irecv {err}, MPI_Isend {err2}, MPI_Waitall {err3}")
    return s["dst"]


class _Graph:
    """The graph communicator and types of one exchange, freed with it."""

    def __init__(self, case):
        self.mpi = tmpi.get()
        self.send = [_commit(_halo_region(case, d, False))[0] for d in DIRECTIONS]
        self.recv = [_commit(_halo_region(case, tuple(-x for x in d), True))[0]
                     for d in DIRECTIONS]
        self.comm = self.mpi.dist_graph([0] * 26, [0] * 26)

    def __del__(self):
        self.mpi.comm_free(self.comm)
        for h in self.send + self.recv:
            self.mpi.free(h)


def _neighbor_prepare(case, seed):
    sub = (case["n"] + 2 * case["radius"]) ** 3 * case["cell"]
    return {"run": _neighbor_run, "graph": _Graph(case), "src": _random_bytes(sub, seed),
            "dst": _filled(sub), "ones": [1] * 26, "zeros": [0] * 26}


def _neighbor_run(s):
    g, ones, zeros = s["graph"], s["ones"], s["zeros"]
    err = g.mpi.neighbor_alltoallw(s["src"].data_ptr(), ones, zeros, g.send, s["dst"].data_ptr(),
                                   ones, zeros, g.recv, g.comm)
    if err:
        raise RuntimeError(f"MPI_Neighbor_alltoallw {err}")
    return s["dst"]


_PREPARE = {"mpi": _mpi_prepare, "stream": _stream_prepare, "faces": _faces_prepare,
            "halo": _halo_prepare, "random": _random_prepare, "sendrecv": _sendrecv_prepare,
            "neighbor": _neighbor_prepare}
_PACKED = {"mpi": _mpi_packed, "stream": _stream_packed, "faces": _faces_packed,
           "halo": _halo_packed, "random": _random_packed, "sendrecv": _sendrecv_packed,
           "neighbor": _halo_bytes}
