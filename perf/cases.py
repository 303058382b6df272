"""The timed workloads of the search framework, each through its public entry points.

Three kinds of work: "device" searches with queries and results resident in HBM
(`NativeIndex.search_dev`, what a serving process on the GPU calls), "host" searches with numpy
arrays (`TurboQuantIndex.search`, `IdMapIndex.search`, with PCIe copies and argument checks inside
the call), and ingest (`add` from host rows up to the snapshot image, `add_dev` from device rows).

Sizes are those of this repository's configurations and benchmark (100K x 128, 1M and 10M x 1536,
3072-dimensional id maps) or generic; `draw` spreads over the same ranges.  Rows are unit vectors:
independent Gaussian, or a mixture of 1000 clusters whose queries lie next to stored rows.
"""
import math

import numpy as np
import torch

from turbovec_amd import _lib as T
from turbovec_amd.index import IdMapIndex, TurboQuantIndex

_CHUNK_FLOATS = 1 << 28          # rows are made and encoded in pieces of 1 GiB
_ADD_ROWS = 100_000              # rows per add of the ingest cases
_MAX_COORDS = 10_000_000 * 1536  # the largest index of the range
_MAX_PRODUCTS = 10_000_000 * 1536 * 1024


def listed():
    return [
        # One user query against a small collection through the Python surface: all latency.
        dict(name="one_100k_128", kind="host", n=100_000, dim=128, bits=4, nq=1, k=10),
        # The small benchmark: a thousand queries in one call on the same collection.
        dict(name="thousand_100k_128", kind="host", n=100_000, dim=128, bits=4, nq=1000, k=10),
        # A serving process that gathers its callers' requests into middle-sized batches.
        dict(name="batch64_1m", kind="device", n=1_000_000, dim=1536, bits=4, nq=64, k=10),
        # Interactive search over the headline collection: one pass over 7.7 GB of codes.
        dict(name="one_10m", kind="device", n=10_000_000, dim=1536, bits=4, nq=1, k=10),
        # The headline batch.
        dict(name="batch_10m", kind="device", n=10_000_000, dim=1536, bits=4, nq=1024, k=10),
        # Interactive search over the compact (2-bit) form of it, a hundred candidates for a re-ranker.
        dict(name="one_10m_2bit", kind="device", n=10_000_000, dim=1536, bits=2, nq=1, k=100),
        # The same as an offline batch: candidates of a thousand queries.
        dict(name="batch_10m_2bit", kind="device", n=10_000_000, dim=1536, bits=2, nq=1024, k=100),
        # Metadata filter that half of a clustered collection passes; a batch size off every tile edge.
        dict(name="masked_4m_768", kind="device", n=4_000_000, dim=768, bits=4, nq=300, k=10, allowed=0.5, data="mixture"),
        # Odd everything, on an index with a fitted calibration; 3-bit codes.
        dict(name="ragged_3bit", kind="device", n=777_777, dim=1000, bits=3, nq=37, k=33, calibrated=True),
        # Id-addressed search restricted to 1 % of the ids, long rows, host arrays in and out.
        dict(name="allowlist_200k_3072", kind="idmap", n=200_000, dim=3072, bits=4, nq=1024, k=10, allowed=0.01),
        # A shard built from an array of embeddings and serialised for storage.
        dict(name="ingest_host", kind="ingest_host", n=100_000, dim=1536, bits=4),
        # Rows produced on the GPU, added to a new index in pieces of 100K.
        dict(name="ingest_device", kind="ingest_device", n=400_000, dim=1536, bits=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    dim = rng.choice([128, 256, 384, 512, 768, 1024, 1536, 2048, 3072]) if rng.random() < 0.5 else 8 * _log_int(rng, 8, 384)
    bits = rng.choice([2, 3, 4, 4])
    what = rng.random()
    if what < 0.12:
        most = 400_000 * 1536 // dim
        return dict(kind="ingest_device", n=_log_int(rng, 1000, min(1_000_000, most)), dim=dim, bits=bits)
    if what < 0.18:
        most = 100_000 * 1536 // dim
        return dict(kind="ingest_host", n=_log_int(rng, 1000, min(100_000, most)), dim=dim, bits=bits)
    nq = 1 if rng.random() < 0.25 else _log_int(rng, 2, 1024)
    k = _log_int(rng, 1, 100)
    if what < 0.28:
        n = _log_int(rng, 5_000, min(400_000, 200_000 * 3072 // dim))
        return dict(kind="idmap", n=n, dim=dim, bits=rng.choice([2, 4]), nq=nq, k=k, allowed=rng.choice([0.01, 0.2]))
    case = dict(kind="device", n=0, dim=dim, bits=bits, nq=nq, k=k)
    most = min(10_000_000, _MAX_COORDS // dim)
    if what < 0.4:
        case["kind"] = "host"
        most = min(most, 400_000 * 256 // dim)
    # 3-bit codes take as many bytes as 4-bit ones and the table scan's time per byte
    most = min(most, _MAX_PRODUCTS // (dim * nq * (2 if bits == 3 else 1)))
    case["n"] = _log_int(rng, 5_000, max(5_001, most))
    if rng.random() < 0.3:
        case["allowed"] = rng.choice([0.5, 0.1, 0.01])
    if rng.random() < 0.3:
        case["data"] = "mixture"
    if case["kind"] == "device" and rng.random() < 0.2:
        case["calibrated"] = True
    return case


class _Rows:
    """Unit rows of one distribution, made on the GPU from a seed."""

    def __init__(self, case, seed):
        self.dim = case["dim"]
        self.g = torch.Generator(device="cuda").manual_seed(seed * 1_000_003 + 17)
        self.centres = None
        if case.get("data") == "mixture":
            self.centres = torch.randn(1000, self.dim, generator=self.g, device="cuda")

    def make(self, rows):
        x = torch.randn(rows, self.dim, generator=self.g, device="cuda")
        if self.centres is not None:
            which = torch.randint(0, len(self.centres), (rows,), generator=self.g, device="cuda")
            x.mul_(0.3).add_(self.centres[which])
        return x.div_(x.norm(dim=1, keepdim=True))

    def queries(self, nq, near):
        """Gaussian data: more of the same; clustered data: stored rows with a little noise."""
        if self.centres is None:
            return self.make(nq)
        which = torch.randint(0, len(near), (nq,), generator=self.g, device="cuda")
        x = near[which] + 0.05 / math.sqrt(self.dim) * torch.randn(nq, self.dim, generator=self.g, device="cuda")
        return x.div_(x.norm(dim=1, keepdim=True))


def _native_index(case, rows):
    """The filled index and its first rows."""
    ix = T.NativeIndex(case["dim"], case["bits"])
    if case.get("calibrated"):
        ix.calibrate(rows.make(2048).cpu().numpy())
    first, done, step = None, 0, max(1, _CHUNK_FLOATS // case["dim"])
    while done < case["n"]:
        x = rows.make(min(step, case["n"] - done))
        torch.cuda.synchronize()
        ix.add_dev(x.data_ptr(), len(x))
        done += len(x)
        if first is None:
            first = x[:4096].clone()
    return ix, first


def prepare(case, seed):
    rows = _Rows(case, seed)
    if case["kind"] == "ingest_host":
        return dict(case=case, rows=rows.make(case["n"]).cpu().numpy())
    if case["kind"] == "ingest_device":
        x = rows.make(case["n"])
        torch.cuda.synchronize()
        return dict(case=case, rows=x)
    rng = np.random.default_rng(seed)
    n, nq = case["n"], case["nq"]
    k_eff = min(case["k"], n)
    if case["kind"] == "device":
        ix, first = _native_index(case, rows)
        state = dict(case=case, index=ix, queries=rows.queries(nq, first), mask=None, n_allowed=0)
        if "allowed" in case:
            words, n_allowed = T.pack_mask(rng.random(n) < case["allowed"])
            state["mask"] = torch.from_numpy(words.view(np.int64)).cuda()
            state["n_allowed"] = n_allowed
            k_eff = min(k_eff, n_allowed)
        state["scores"] = torch.empty(nq, k_eff, dtype=torch.float32, device="cuda")
        state["slots"] = torch.empty(nq, k_eff, dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
        return state
    # host kinds: an index loaded from its snapshot image, as a service starts
    ix, first = _native_index(case, rows)
    state = dict(case=case, queries=rows.queries(nq, first).cpu().numpy(), mask=None)
    if case["kind"] == "idmap":
        ids = rng.permutation(np.arange(n, dtype=np.uint64) * np.uint64(2_654_435_761) + np.uint64(seed & 0xFFFF))
        state["index"] = IdMapIndex.from_bytes(ix.to_bytes(ids=ids))
        state["allowlist"] = rng.choice(ids, max(1, int(case["allowed"] * n)), replace=False)
    else:
        state["index"] = TurboQuantIndex.from_bytes(ix.to_bytes())
        if "allowed" in case:
            state["mask"] = rng.random(n) < case["allowed"]
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "device":
        mask = state["mask"]
        state["index"].search_dev(state["queries"].data_ptr(), case["nq"], case["k"], state["scores"].data_ptr(),
                                  state["slots"].data_ptr(), None if mask is None else mask.data_ptr(), state["n_allowed"])
        return state["scores"], state["slots"]
    if kind == "host":
        return state["index"].search(state["queries"], case["k"], mask=state["mask"])
    if kind == "idmap":
        scores, ids = state["index"].search(state["queries"], case["k"], allowlist=state["allowlist"])
        return scores, ids.view(np.int64)
    if kind == "ingest_host":
        index = TurboQuantIndex(case["dim"], case["bits"])
        index.add(state["rows"])
        return np.frombuffer(index.to_bytes(), np.uint8)
    index = T.NativeIndex(case["dim"], case["bits"])
    rows = state["rows"]
    for at in range(0, case["n"], _ADD_ROWS):
        piece = rows[at:at + _ADD_ROWS]
        index.add_dev(piece.data_ptr(), len(piece))
    codes, scales, code_bytes = index.device_ptrs()
    return _view(index, codes, code_bytes, "|u1"), _view(index, scales, case["n"], "<f4")


class _Device:
    """Device memory of an index; a tensor made from it holds this object, and this object the index."""

    def __init__(self, index, ptr, count, kind):
        self.index = index
        self.__cuda_array_interface__ = dict(shape=(count,), typestr=kind, data=(ptr, False), version=2)


def _view(index, ptr, count, kind):
    return torch.as_tensor(_Device(index, ptr, count, kind), device="cuda")


def work(case):
    """What the task itself needs: the allowed rows' codes and scales, the queries, the results; one
    multiply-add per dimension of every (query, allowed row) pair.  Ingest reads the rows and writes
    codes and scales; its arithmetic is the two rounds of butterflies and the norm."""
    n, dim = case["n"], case["dim"]
    row = dim * (2 if case["bits"] == 2 else 4) // 8 + 4
    if case["kind"].startswith("ingest"):
        return {"bytes": n * (4 * dim + row), "flops": n * dim * (2 * math.log2(dim & -dim) + 2)}
    rows = n * case.get("allowed", 1.0)
    nq, k = case["nq"], min(case["k"], n)
    return {"bytes": rows * row + ("allowed" in case) * n / 8 + nq * (4 * dim + 12 * k), "flops": 2.0 * nq * rows * dim}


def tolerance(case):
    """Integer sums over integer tables, one stated order of the float operations around them, a total
    order on results: every correct implementation returns the same bits."""
    return "exact"
