"""The work a program has this library do, as cases that can be timed and checked.

A case is a dict of plain values.  Its "kind" is the call it makes:

  share      Faces.share(u, compute): one exchange + DSS step of one field
  transport  the staged pieces a program with its own transport calls:
             pack, exchange (device copies in the transport's place),
             inner_unpack
  six        Faces.share on the 6-message schedule
  batch      Batch.share: many independent grids in one call
  serve      Server.submit and Server.wait: requests handed over at once

Fields are float64 and stepped in place; what a pass returns is the field (for
batch and serve the one buffer that holds every grid's field).  Results are
compared exactly: the order of every node's sum is part of the interface.
"""
import math
import random

import numpy as np
import torch

import faces_amd as fa

GRID_PAD = 64  # doubles: each grid of a batch starts on 512 bytes, as an allocation of its own would


def _one(kind, n, mx, my, mz, ranks=(1, 1, 1), rank=0, boundary="periodic", compute=True, padded=False, data="random", name=None):
    c = {"kind": kind, "n": n, "mx": mx, "my": my, "mz": mz, "lx": ranks[0], "ly": ranks[1], "lz": ranks[2], "rank": rank,
         "boundary": boundary, "compute": compute, "padded": padded, "data": data}
    return dict(c, name=name) if name else c


def _many(kind, grids, low, high, orders, mix, name=None):
    c = {"kind": kind, "grids": grids, "low": low, "high": high, "orders": orders, "mix": mix, "boundary": "periodic"}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call, a test-size field: launch and call latency
        _one("share", 5, 4, 4, 4, data="int", name="share_4x4x4_n5"),
        # the reference's small run line, its own boundary mode and page-padded planes: one rank per GPU, 10,000 shares
        _one("share", 12, 15, 14, 13, boundary="open", padded=True, name="share_15x14x13_n12_open_padded"),
        # one rank of a 6x6x6 decomposition, random data
        _one("share", 8, 32, 32, 32, name="share_32x32x32_n8"),
        # the benchmark's step
        _one("share", 7, 60, 60, 60, data="int", name="share_60x60x60_n7"),
        # rows, columns and planes of prime length at low order
        _one("share", 3, 127, 61, 97, name="share_127x61x97_n3"),
        # a high polynomial order (degree 15)
        _one("share", 16, 24, 20, 17, name="share_24x20x17_n16"),
        # the reference's large run line: 11.5 GB, offsets beyond 32 bits
        _one("share", 12, 95, 94, 93, boundary="open", padded=True, name="share_95x94x93_n12_open_padded"),
        # communication only (compute = 0): a corner rank sums its surface and leaves its interior
        _one("share", 8, 40, 44, 42, ranks=(2, 2, 2), boundary="open", compute=False, name="surface_40x44x42_n8_corner"),
        # an interior rank whose messages a transport carries
        _one("transport", 7, 60, 60, 60, ranks=(3, 3, 3), rank=13, boundary="open", name="transport_60x60x60_n7_interior"),
        # the 6-message schedule on a rank with neighbours on some sides
        _one("six", 6, 48, 50, 52, ranks=(3, 2, 2), rank=4, boundary="open", name="six_48x50x52_n6_edge"),
        # many small grids of uneven sizes stepped together
        _many("batch", 256, 2, 24, "4,6,8", 4, name="batch_256_mixed"),
        # a burst of requests to the server
        _many("serve", 64, 2, 24, "4,6,8", 5, name="serve_64_mixed"),
    ]


def draw(rng):
    u = rng.random()
    if u < 0.14:
        return _many("batch", round(math.exp(rng.uniform(math.log(4), math.log(300)))), 1, rng.randint(6, 28),
                     rng.choice(["4,6,8", "5,7", "3,4,5", "6,8,9,10", "2,8,12"]), rng.randrange(1 << 20))
    if u < 0.22:
        return _many("serve", round(math.exp(rng.uniform(math.log(2), math.log(100)))), 1, rng.randint(6, 24),
                     rng.choice(["4,6,8", "5,7", "3,4,5", "6,8,9,10"]), rng.randrange(1 << 20))
    n = rng.choice([2, 3, 4, 4, 5, 5, 6, 6, 7, 7, 8, 8, 9, 10, 11, 12, 12, 13, 14, 16])
    elements = math.exp(rng.uniform(math.log(64e3), math.log(2.5e9))) / (8 * n ** 3)
    side = max(1.0, elements) ** (1 / 3)
    m = [max(1, round(side * math.exp(rng.uniform(-0.4, 0.4)))) for _ in range(3)]
    kind = "share" if u < 0.70 else "transport" if u < 0.86 else "six"
    boundary = "open" if kind == "transport" else rng.choice(["periodic", "periodic", "open"])
    ranks, rank = (1, 1, 1), 0
    if boundary == "open" and (kind == "transport" or rng.random() < 0.7):
        ranks = (rng.randint(1, 3), rng.randint(1, 3), rng.randint(2, 3))
        rank = rng.randrange(ranks[0] * ranks[1] * ranks[2])
    compute = kind != "share" or rng.random() < 0.75
    return _one(kind, n, *m, ranks=ranks, rank=rank, boundary=boundary, compute=compute, padded=rng.random() < 0.3,
                data=rng.choice(["int", "random"]))


def _stride(case):
    """Doubles from one plane of elements to the next: dense, or padded to whole pages of 4096 bytes."""
    dense = case["n"] ** 3 * case["mx"] * case["my"]
    return -(-dense // 512) * 512 if case["padded"] else dense


def _grids(case):
    """Sizes (n, mx, my, mz) and starts of the grids of a batch, and the doubles they take together."""
    rng = random.Random(case["mix"])
    orders = [int(n) for n in case["orders"].split(",")]
    shapes = [(rng.choice(orders), *(rng.randint(case["low"], case["high"]) for _ in range(3))) for _ in range(case["grids"])]
    starts, at = [], 0
    for n, mx, my, mz in shapes:
        starts.append(at)
        at += -(-n ** 3 * mx * my * mz // GRID_PAD) * GRID_PAD
    return shapes, starts, at


def _inputs(case, seed):
    """The field, or the buffer that holds every grid's field."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    if case["kind"] in ("batch", "serve"):
        return torch.empty(_grids(case)[2], dtype=torch.float64, device="cuda").uniform_(-1, 1, generator=g)
    dense, ps, mz = case["n"] ** 3 * case["mx"] * case["my"], _stride(case), case["mz"]
    u = torch.zeros(ps * (mz - 1) + dense, dtype=torch.float64, device="cuda")
    nodes = u.as_strided((mz, dense), (ps, 1))
    if case["data"] == "int":
        nodes.random_(0, 1024, generator=g)
    else:
        nodes.uniform_(-1, 1, generator=g)
    return u


_server = None


def _the_server():
    """A program has one server, which outlives its requests."""
    global _server
    if _server is None:
        _server = fa.Server(footprint_cap=100e9, max_batch=256, nstreams=2)
    return _server


def prepare(case, seed):
    u = _inputs(case, seed)
    state = {"kind": case["kind"], "u": u}
    boundary = fa.OPEN if case["boundary"] == "open" else fa.PERIODIC
    if case["kind"] in ("batch", "serve"):
        shapes, starts, _ = _grids(case)
        fields = [u[at:at + n ** 3 * mx * my * mz] for (n, mx, my, mz), at in zip(shapes, starts)]
        if case["kind"] == "batch":
            state["batch"] = fa.Batch(shapes, boundary=boundary)
            state["batch"].set_fields(fields)
        else:
            state["server"], state["requests"] = _the_server(), list(zip(fields, shapes))
            torch.cuda.synchronize()  # a field is ready when it is submitted
        return state
    f = fa.Faces(case["rank"], case["lx"], case["ly"], case["lz"], case["mx"], case["my"], case["mz"], case["n"],
                 boundary=boundary, plane_stride=_stride(case) if case["padded"] else 0)
    if case["kind"] == "six":
        f.set_path(fa.PATH_SIX)
    state["faces"], state["compute"] = f, case["compute"]
    return state


def run(state):
    u = state["u"]
    if state["kind"] == "batch":
        state["batch"].share()
    elif state["kind"] == "serve":
        server = state["server"]
        tickets = [server.submit(field, *shape) for field, shape in state["requests"]]
        for ticket in tickets:
            server.wait(ticket)
    elif state["kind"] == "transport":
        f = state["faces"]
        f.pack(u)
        f.exchange()
        f.inner_unpack(u)
    else:
        state["faces"].share(u, state["compute"])
    return u


def _neighbours(case):
    """Per axis x, y, z: whether there is a neighbour on the low and on the high side."""
    if case["boundary"] == "periodic":
        return [(True, True)] * 3
    at = (case["rank"] % case["lx"], case["rank"] // case["lx"] % case["ly"], case["rank"] // (case["lx"] * case["ly"]))
    return [(k > 0, k < m - 1) for k, m in zip(at, (case["lx"], case["ly"], case["lz"]))]


def _touched(case):
    """Lines of 64 bytes that hold a node the step changes: memory moves no less than a line."""
    n, (mx, my, mz) = case["n"], (case["mx"], case["my"], case["mz"])
    sides = _neighbours(case)

    def axis(j, m, side):  # of the n points of element j: which are shared along this axis, and which lie on the rank's surface
        shared, surface = np.zeros(n, bool), np.zeros(n, bool)
        shared[0], shared[n - 1] = j > 0 or side[0], j < m - 1 or side[1]
        surface[0], surface[n - 1] = j == 0, j == m - 1
        return shared, surface

    x = [np.array(v)[None, :, None, None, :] for v in zip(*(axis(j, mx, sides[0]) for j in range(mx)))]
    y = [np.array(v)[:, None, None, :, None] for v in zip(*(axis(j, my, sides[1]) for j in range(my)))]

    def plane(jz):
        z = [v[None, None, :, None, None] for v in axis(jz, mz, sides[2])]
        nodes = x[0] | y[0] | z[0]
        if not case["compute"]:
            nodes = nodes & (x[1] | y[1] | z[1])
        nodes = nodes.reshape(-1)
        return int(np.pad(nodes, (0, -nodes.size % 8)).reshape(-1, 8).any(1).sum())

    return plane(0) + (plane(mz - 1) if mz > 1 else 0) + (max(0, mz - 2) * plane(mz // 2) if mz > 2 else 0)


def work(case):
    """Each touched line read once and written once, and each message; the additions are one fewer than the copies of each node."""
    if case["kind"] in ("batch", "serve"):
        total = {"bytes": 0, "flops": 0}
        for shape in _grids(case)[0]:
            w = work(_one("share", *shape))
            total = {k: total[k] + w[k] for k in total}
        return total
    n, m = case["n"], (case["mx"], case["my"], case["mz"])
    bytes_ = 2 * 64 * _touched(case)
    if case["kind"] == "transport" or not case["compute"]:
        pairs = [(lo + hi) for lo, hi in _neighbours(case)]  # faces with a neighbour, whose messages are written and read
        bytes_ += 2 * 8 * n * n * (pairs[0] * m[1] * m[2] + pairs[1] * m[0] * m[2] + pairs[2] * m[0] * m[1])
    if case["compute"]:
        adds = n ** 3 * math.prod(m) - math.prod(k * (n - 1) for k in m)
    else:
        adds = 2 * n * n * (m[0] * m[1] + m[1] * m[2] + m[0] * m[2])
    return {"bytes": bytes_, "flops": adds}


def tolerance(case):
    # every node's copies are added in one documented order, so that two correct implementations agree bit for bit
    return "exact"


def _sum_pairs(v, axis, sides):
    """v[jz, jy, jx, iz, iy, ix]: sums the copies that are neighbours along an axis (0 x, 1 y, 2 z); across the rank's surface the
    neighbour's copy is this rank's own from the opposite side."""
    el, node, m = 2 - axis, 5 - axis, v.shape[2 - axis]
    low, high = v.select(node, 0), v.select(node, v.shape[node] - 1)
    first, last = low.select(el, 0), high.select(el, m - 1)
    across = first + last
    if m > 1:
        inner = high.narrow(el, 0, m - 1) + low.narrow(el, 1, m - 1)
        high.narrow(el, 0, m - 1).copy_(inner)
        low.narrow(el, 1, m - 1).copy_(inner)
    if sides[0]:
        first.copy_(across)
    if sides[1]:
        last.copy_(across)


def _share(v, case):
    sides = _neighbours(case)
    full = v if case["compute"] else v.clone()
    for axis in (2, 1, 0) if case["kind"] == "six" else (0, 1, 2):
        _sum_pairs(full, axis, sides[axis])
    if not case["compute"]:  # only the rank's surface
        for axis in range(3):
            el, node = 2 - axis, 5 - axis
            for j, i in ((0, 0), (v.shape[el] - 1, v.shape[node] - 1)):
                v.select(node, i).select(el, j).copy_(full.select(node, i).select(el, j))


def exact(case, seed):
    u = _inputs(case, seed)
    if case["kind"] in ("batch", "serve"):
        shapes, starts, _ = _grids(case)
        for (n, mx, my, mz), at in zip(shapes, starts):
            _share(u[at:at + n ** 3 * mx * my * mz].view(mz, my, mx, n, n, n), _one("share", n, mx, my, mz))
        return u
    n, mx, my, mz = case["n"], case["mx"], case["my"], case["mz"]
    _share(u.as_strided((mz, my, mx, n, n, n), (_stride(case), n ** 3 * mx, n ** 3, n * n, n, 1)), case)
    return u
