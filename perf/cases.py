"""The snapshot dataplane's measured work: saves, restores and device-side record moves at the sizes users run.

A case is one call (or one pair of calls) a serving program makes on a registered plane, from a turn's single block
on one tensor-parallel rank to a whole 8k-token session.  Geometries are the models this repository's benchmark and
tests use (Qwen3-8B, 36 layers; Qwen3-1.7B, 28 layers; 8 KV heads of 128, bf16 or fp8, whole or a tensor-parallel
rank's heads) and generic odd ones.  Every output is bytes or whole numbers, so every tolerance is exact.

What the kinds stand for:

* ``save``: ``save_gather`` of a session's blocks into pinned records, with or without the digests that name its
  blobs; a hashed save is over when its ids are there.
* ``restore``: ``load_scatter`` (or ``load_scatter_checked``) of pinned records into newly allocated blocks.
* ``disk``: ``load_from_disk`` of a snapshot's blob files, every CRC32C checked on the GPU.
* ``move``: ``gather_blocks`` then ``scatter_blocks``, a session's records packed in device memory and placed in
  other blocks.
"""
from __future__ import annotations

import ctypes
import random
import shutil
import tempfile

import numpy as np
import torch

from kvsnap_amd.blobs import BlobDirectory
from kvsnap_amd.crc32c import crc32c
from kvsnap_amd.dataplane import TorchBlockDataPlane, gather_blocks, scatter_blocks

QWEN3_8B = dict(layers=36, heads=8, head_dim=128, dtype="bf16", block_size=16)
QWEN3_8B_TP8 = dict(QWEN3_8B, heads=1)
QWEN3_8B_TP4 = dict(QWEN3_8B, heads=2)
QWEN3_8B_TP2 = dict(QWEN3_8B, heads=4)
QWEN3_1_7B = dict(layers=28, heads=8, head_dim=128, dtype="bf16", block_size=16)
QWEN3_1_7B_FP8 = dict(QWEN3_1_7B, dtype="fp8")
#: A generic model whose spans are neither whole KiB nor powers of two.
ODD = dict(layers=25, heads=3, head_dim=80, dtype="bf16", block_size=16)

SAVE = dict(kind="save", mode="staged", hashed=False)
RESTORE = dict(kind="restore", mode="dma", checked=False)
#: No case moves more than the 8k-token Qwen3-8B session's records.
LARGEST = 512 * 2359296
#: Blob files are written for each preparation, so disk restores stay smaller.
LARGEST_DISK = 256 << 20


def listed():
    return [
        # Latency: the one block a short reply filled, on one of eight ranks; its tail is not filled.
        dict(SAVE, **QWEN3_8B_TP8, name="save-one-block-tp8", layout="vllm", tokens=11),
        # Latency: a short prompt's blocks back into the cache.
        dict(RESTORE, **QWEN3_1_7B_FP8, name="restore-5-blocks-fp8", layout="vllm", tokens=80),
        # A turn of about 512 tokens added to a session: what a delta save gathers and hashes.
        dict(SAVE, **QWEN3_8B, name="save-hashed-turn", layout="vllm", tokens=507, hashed=True),
        # The whole 8k-token session, hashed: the largest save.
        dict(SAVE, **QWEN3_8B, name="save-hashed-8k", layout="kv_split", tokens=8192, hashed=True),
        # The same session on one of eight ranks.
        dict(SAVE, **QWEN3_8B_TP8, name="save-hashed-8k-tp8", layout="vllm", tokens=8185, hashed=True),
        # A session saved beside a decode: the kernel writes pinned memory itself.
        dict(SAVE, **QWEN3_1_7B_FP8, name="save-direct-hashed-2k-fp8", layout="kv_split", tokens=2048,
             mode="direct", hashed=True),
        # An ordinary save whose ids are taken elsewhere, spans of 7,680 bytes, a ragged tail.
        dict(SAVE, **ODD, name="save-4k-odd", layout="kv_split", tokens=3999),
        # The whole session back through the copy engines: the largest restore.
        dict(RESTORE, **QWEN3_8B, name="restore-8k", layout="kv_split", tokens=8192),
        # An ordinary restore with its checksums compared.
        dict(RESTORE, **QWEN3_1_7B, name="restore-checked-2k", layout="vllm", tokens=2048, checked=True),
        # The restore kernel reading pinned memory in place, on one of four ranks.
        dict(RESTORE, **QWEN3_8B_TP4, name="restore-kernel-1k-tp4", layout="vllm", tokens=1000, mode="kernel"),
        # A snapshot's blob files back into the cache.
        dict(QWEN3_1_7B, name="restore-disk-2k", kind="disk", layout="vllm", tokens=2048),
        # Device memory only: an 8k-token session's records packed and placed on one of two ranks.
        dict(QWEN3_8B_TP2, name="move-8k-tp2", kind="move", layout="kv_split", tokens=8192),
    ]


def draw(rng):
    kind = rng.choice(["save", "save", "save", "restore", "restore", "restore", "disk", "move"])
    case = dict(kind=kind, layout=rng.choice(["vllm", "kv_split"]), block_size=rng.choice([16, 16, 32]),
                layers=rng.randint(2, 40), heads=rng.choice([1, 2, 3, 4, 5, 8]),
                head_dim=rng.choice([64, 80, 96, 112, 128]), dtype=rng.choice(["bf16", "fp8"]))
    if kind == "save":
        case.update(mode=rng.choice(["staged", "staged", "direct"]), hashed=rng.random() < 0.6)
    elif kind == "restore":
        case.update(mode=rng.choice(["dma", "dma", "kernel"]), checked=rng.random() < 0.5)
    while record_bytes(case) > 2359296:             # a record's hash is one chain: no longer than the listed ones
        case["layers"] = rng.randint(2, 30)
        case["heads"] = rng.choice([1, 2, 3, 4])
    most = (LARGEST_DISK if kind == "disk" else LARGEST // 2 if kind == "move" else LARGEST) // record_bytes(case)
    blocks = round(min(most, 2048) ** rng.random())
    case["tokens"] = max(1, blocks * case["block_size"] - rng.choice([0, rng.randrange(case["block_size"])]))
    return case


def record_bytes(case):
    element = 2 if case["dtype"] == "bf16" else 1
    return 2 * case["layers"] * case["heads"] * case["head_dim"] * case["block_size"] * element


def work(case):
    """A save reads the blocks and writes the records, a restore the inverse; a move does both in turn."""
    once = blocks_of(case) * record_bytes(case)
    return {"bytes": (4 if case["kind"] == "move" else 2) * once, "flops": 0}


def tolerance(case):
    return "exact"


def blocks_of(case):
    return -(-case["tokens"] // case["block_size"])


class Plane:
    """A registered plane, closed (its pinned arena freed) once nothing refers to it or to its pinned bytes."""

    def __init__(self, caches, case, capacity):
        self.plane = TorchBlockDataPlane(caches, case["block_size"], capacity,
                                         save_mode=case["mode"] if case["kind"] == "save" else None,
                                         restore_mode=case["mode"] if case["kind"] == "restore" else None)

    def pinned(self, nbytes):
        """A reservation of the plane's pool, and its bytes as a tensor that keeps this plane open."""
        staged = self.plane.pool.reserve(nbytes)
        view = type("Pinned", (ctypes.c_uint8 * nbytes,), {}).from_address(staged.pointer)
        view.plane = self
        return staged, torch.from_numpy(np.ctypeslib.as_array(view))

    def __del__(self):
        if hasattr(self, "plane"):
            self.plane.close()


class Session:
    """A registered plane, a session's block table and its pinned records (and blob files)."""

    def __init__(self, case, seed):
        self.case, self.n, self.size = case, blocks_of(case), record_bytes(case)
        rng = random.Random(seed)
        total = 2 * self.n + 9
        ids = rng.sample(range(1, total), 2 * self.n)
        self.source, self.target = ids[:self.n], ids[self.n:]
        gen = torch.Generator("cuda")
        gen.manual_seed(seed)
        self.caches, self.backing = make_caches(case, total, gen)
        chunk = max(1, min(self.n, (128 << 20) // self.size))     # load_from_disk's ring: up to four 128 MiB chunks
        ring = min(4, -(-self.n // chunk)) * chunk * self.size if case["kind"] == "disk" else 0
        self.owner = Plane(self.caches, case, self.n * self.size + ring + (1 << 20))
        self.plane = self.owner.plane
        self.plane.warm_up()
        self.root = None
        self.staged, records = self.owner.pinned(self.n * self.size)
        self.records = records.view(self.n, self.size)
        self.slots = [(self.staged, i * self.size) for i in range(self.n)]
        if case["kind"] == "restore":
            self.records.copy_(values((self.n, self.size), case["dtype"], gen))
            if case["checked"]:
                self.crcs = [crc32c(record.numpy().tobytes()) for record in self.records]
        elif case["kind"] == "disk":
            self.root = tempfile.mkdtemp(prefix="kvsnap-cases-")
            self.blobs = BlobDirectory(self.root)
            digests = []
            self.plane.save_gather(self.source, self.slots, case["tokens"], digests=digests)
            self.segments = self.blobs.write_blocks(
                [(self.staged.pointer + i * self.size, self.size) for i in range(self.n)], digests[0].result())
        elif case["kind"] == "move":
            spans = self.plane.spans()
            columns = ([s[0] for s in spans], [s[1] for s in spans], [s[2] for s in spans],
                       [s[3] // 8 for s in spans], self.source, self.target)
            *self.tables, self.from_ids, self.to_ids = [torch.tensor(c, dtype=torch.int64, device="cuda")
                                                        for c in columns]
            self.shortest = min(s[3] for s in spans)
            self.packed = torch.empty((self.n, self.size), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()

    def __del__(self):
        if getattr(self, "root", None):
            shutil.rmtree(self.root, ignore_errors=True)


def values(shape, dtype, gen):
    """KV-like bytes: N(0, 1) elements of the cache's type, as uint8."""
    *lead, last = shape
    if dtype == "bf16":
        return torch.randn((*lead, last // 2), dtype=torch.bfloat16, device="cuda", generator=gen).view(torch.uint8)
    out = torch.empty(shape, dtype=torch.uint8, device="cuda")
    for row in out:                                  # row by row: the 32-bit intermediates stay small
        row.copy_(torch.randn(row.shape, device="cuda", generator=gen).to(torch.float8_e4m3fn).view(torch.uint8))
    return out


def make_caches(case, total, gen):
    """Every layer's cache view, carved from one allocation of uint8 values."""
    dtype = torch.bfloat16 if case["dtype"] == "bf16" else torch.float8_e4m3fn
    layers, heads, dim, tokens = case["layers"], case["heads"], case["head_dim"], case["block_size"]
    element = 2 if case["dtype"] == "bf16" else 1
    if case["layout"] == "vllm":                     # [blocks, heads, tokens, 2 * dim] views of token-major storage
        shape = (layers, total, tokens, heads, 2 * dim)
        backing = values((*shape[:-1], 2 * dim * element), case["dtype"], gen)
        caches = [backing[i].view(dtype).permute(0, 2, 1, 3) for i in range(layers)]
    else:                                            # K and V apart: [2, blocks, tokens, heads, dim]
        shape = (layers, 2, total, tokens, heads, dim)
        backing = values((*shape[:-1], dim * element), case["dtype"], gen)
        caches = [backing[i].view(dtype) for i in range(layers)]
    return {f"model.layers.{i}.self_attn.attn": cache for i, cache in enumerate(caches)}, backing


def prepare(case, seed):
    return Session(case, seed)


def run(state):
    case, plane = state.case, state.plane
    if case["kind"] == "save":
        digests = [] if case["hashed"] else None
        plane.save_gather(state.source, state.slots, case["tokens"], digests=digests)
        if not case["hashed"]:
            return state.records
        found = digests[0].result()
        return {"records": state.records,
                "sha256": np.frombuffer(bytes.fromhex("".join(sha for sha, _ in found)), dtype=np.uint8),
                "crc32c": np.array([crc for _, crc in found], dtype=np.int64)}
    if case["kind"] == "restore":
        if case["checked"]:
            plane.load_scatter_checked(state.target, state.slots, state.crcs)
        else:
            plane.load_scatter(state.target, state.slots)
    elif case["kind"] == "disk":
        plane.load_from_disk(state.target, state.blobs, state.segments)
    else:
        gather_blocks(state.from_ids, *state.tables, state.packed.data_ptr(), state.size,
                      min_span_bytes=state.shortest)
        scatter_blocks(state.packed.data_ptr(), state.size, state.to_ids, *state.tables,
                       min_span_bytes=state.shortest)
        return {"records": state.packed, "caches": state.backing}
    return state.backing
