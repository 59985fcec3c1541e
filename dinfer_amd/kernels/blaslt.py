"""bf16 matrix products of many rows through hipBLASLt or the tile kernel, whichever a measurement per shape finds faster.

The reference hands these products to its vendor library too (crates/kernels/src/gemm.rs:605-647).
The library's first suggestion is what a framework's own matmul runs; for few output tiles and a long K it is
far off (N 5,120, K 17,408 at 520 rows: 167 us against 102 us for the best of the library's own list),
so here the library is called directly and its candidate list for a shape is timed.

Beside the library's list stand a few shapes of the tile kernel (csrc/gemm_tile.hip; tiles.py names those worth timing), which
also takes what follows a product into its end (`with_end`): timed against the library's product and the pass of its own together, in trains.

When it is timed, and what a product runs with otherwise, is settled so that results repeat:
  * a product outside `measuring()` never times anything: it runs the algorithm its shape was given earlier,
    or the library's first suggestion. The engine's warm-up runs one step of every row count under
    `measuring()`, before it serves; no serving step stalls for a measurement.
  * of the timed candidates the one with the lowest index within TIE of the fastest wins, so two runs that
    time the same candidates a per cent apart choose the same one.
  * the choices are kept in a plan file beside the built libraries, keyed by device, library and shape; a later
    process finds them there, measures nothing and computes the same bits as the one that measured.
  * `configure(tuning="heuristic")` takes the library's first suggestion everywhere (no measurement, no file).
These are engine options (EngineOptions.gemm_tuning, gemm_plan_file), not environment switches. A shape the
library names no algorithm for is left to the caller (`matmul` returns False), who runs the plain kernel.

out[M, N] = a[M, K] . w[N, K]^T in row-major storage is, in the library's column-major terms,
D (N x M, ld = ldc) = op_T(w as K x N, ld = ldw) . (a as K x M, ld = lda).
"""
from __future__ import annotations

import contextlib
import ctypes
import json
import os
import sys
from collections.abc import Callable
from ctypes import POINTER, byref, c_float, c_int, c_int32, c_int64, c_size_t, c_uint64, c_void_p

import torch

from . import ops, tiles

WORKSPACE_BYTES = 128 << 20   # for the library's split-K and stream-K kernels
CANDIDATES = 32               # how many of the library's suggestions are timed (the best has been seen as far down as 21st)
FLUSH_BYTES = 512 << 20       # read before each timed run: twice the memory-side cache
TUNE_FROM_ROWS = 33           # every size that comes here (up to 32 rows the weight-streaming kernel runs)
TUNE_FROM_WORK = 1 << 24      # rows x columns x depth below which no choice of kernel repays its measurement
TIE = 0.03                    # candidates within this fraction of the fastest count as equal: the lowest index wins
# A product with its end in one kernel is timed against the product and its pass in trains: launches of one form back to back, each with another
# copy of the weight. Behind emptied caches a single launch runs at a clock that a step does not have: the library's, bound by the matrix
# cores, take longer in a step than timed alone, the tile kernel, bound by its loads, does not. us, the product and its pass and the tile, alone,
# in trains and in a step: gated 2,048 x 24,576 x 4,096 294 and 291, 306 and 299, 303 and 286; 2,048 x 16,384 x 2,048 118 and 111, 120 and 110, 119
# and 104; 544 x 34,816 x 5,120 195 and 186, 200 and 189, 194 and 182; relu2 4,096 x 8,192 x 2,048 125 and 130, 124 and 116, 120 and 117. Three
# processes with files of their own took the same side at 27 of 28 shapes (512 rows 98 and 96 tile, 1,024 rows 180 and 181 pass; 256 rows, 67
# and 65 to 66, differed).
TRAIN_MS = 5.0                # of one form until its clock has settled, and as long again timed (trains of 3 in turn share a clock: 300 and 301 at the first)
TRAINS = 2                    # of each form
TRAIN_TIE = 0.015             # the product and its pass run where they are within this of the fastest (trains repeat within 1 %)
TRAIN_TILES = 2               # the fastest tile alone, and the next one within 5 % of it
TRAIN_CLEAR = 1.25            # a form this far above the fastest alone is left out (alone and in trains the two sides moved by up to 16 %)

_HIP_R_32F, _HIP_R_16BF = 0, 14
_OP_N, _OP_T = 111, 112
_COMPUTE_32F = 2
_DESC_TRANSA, _DESC_TRANSB = 0, 1
_PREF_MAX_WORKSPACE = 1


class _Algo(ctypes.Structure):
    _fields_ = [("data", ctypes.c_uint8 * 16), ("max_workspace_bytes", c_size_t)]


class _Heuristic(ctypes.Structure):
    _fields_ = [("algo", _Algo), ("workspace_size", c_size_t), ("state", c_int), ("waves_count", c_float),
                ("reserved", c_int * 4)]


_lib = None
_lib_tried = False
_handles: dict = {}
_workspaces: dict = {}
_plans: dict = {}
_flush: dict = {}
_one, _zero = c_float(1.0), c_float(0.0)

# settings of the process (the engine sets them from its options when it is built)
_settings = {"tuning": "measured", "plan_file": None, "log": False}
_measuring = False            # inside measuring(): shapes without a choice are timed
# the plan file's contents: shape key -> {"index": i, "algo": hex of the algorithm's bytes}, with "tile": [rows, columns] where the tile
# kernel was faster than that one; of a product with its end "tile" alone, null for a pass of its own
_stored: dict | None = None
_stored_path = None


def configure(tuning: str | None = None, plan_file=..., log: bool | None = None) -> None:
    """tuning "measured": candidates are timed inside measuring() and the choices kept in the plan file;
    "heuristic": the library's first suggestion for every shape. plan_file: where choices are kept between
    processes ("" for nowhere; None: beside the built libraries; left out: as it was). Arguments left out or None
    (plan_file aside) change nothing. Shapes that already have a plan keep it."""
    global _stored, _stored_path
    if tuning is not None and tuning not in ("measured", "heuristic"):
        raise ValueError(f"gemm tuning must be 'measured' or 'heuristic', got {tuning!r}")
    for k, v in (("tuning", tuning), ("log", log)):
        if v is not None:
            _settings[k] = v
    if plan_file is not ... and plan_file != _settings["plan_file"]:
        _save_stored()
        _settings["plan_file"] = plan_file
        _stored = _stored_path = None
        for plan in (*_plans.values(), *_ends.values()):
            if plan:
                plan.asked = False      # shapes without a choice are looked up in the new file


@contextlib.contextmanager
def measuring():
    """Products of shapes that have no choice yet time their candidates in here (the engine's warm-up)."""
    global _measuring
    before, _measuring = _measuring, _settings["tuning"] == "measured"
    try:
        yield
    finally:
        _measuring = before
        _save_stored()


def _plan_path(dev):
    global _stored_path
    if _stored_path is None:
        f = _settings["plan_file"]
        if f == "":
            return None
        if f is None:
            from ..csrc import build
            import hashlib
            ident = f"{torch.cuda.get_device_name(dev)}|{torch.version.hip}|{CANDIDATES}|{WORKSPACE_BYTES}|trains"
            f = str(build.lib_dir() / f"blaslt_plans_{hashlib.sha256(ident.encode()).hexdigest()[:12]}.json")
        _stored_path = f
    return _stored_path


_stored_dirty = False
worth_measuring_met = 0       # how many products so far were of a size whose algorithm is worth measuring


def _load_stored(dev) -> dict:
    global _stored
    if _stored is None:
        _stored = {}
        path = _plan_path(dev)
        if path and os.path.exists(path):
            try:
                with open(path) as fh:
                    data = json.load(fh)
                if isinstance(data, dict):
                    _stored = data
            except (OSError, ValueError):
                pass   # an unreadable file is measured again and rewritten
    return _stored


def _save_stored() -> None:
    global _stored_dirty
    if not _stored_dirty or _stored is None or not _stored_path:
        return
    _stored_dirty = False
    try:
        # other processes may have added shapes since this one read the file
        merged = {}
        if os.path.exists(_stored_path):
            try:
                with open(_stored_path) as fh:
                    merged = json.load(fh)
            except (OSError, ValueError):
                merged = {}
        merged.update(_stored)
        tmp = f"{_stored_path}.{os.getpid()}.tmp"
        with open(tmp, "w") as fh:
            json.dump(merged, fh, indent=0, sort_keys=True)
        os.replace(tmp, _stored_path)
    except OSError:
        pass   # a folder that cannot be written: the choices live as long as the process


def _load():
    global _lib, _lib_tried
    if _lib_tried:
        return _lib
    _lib_tried = True
    # the copy torch itself has loaded comes first: one instance of the library and of its kernels per process
    for path in (os.path.join(os.path.dirname(torch.__file__), "lib", "libhipblaslt.so"),
                 "/opt/rocm/lib/libhipblaslt.so"):
        if os.path.exists(path):
            try:
                lib = ctypes.CDLL(path)
            except OSError:
                continue
            P = c_void_p
            lib.hipblasLtCreate.argtypes = [POINTER(P)]
            lib.hipblasLtMatmulDescCreate.argtypes = [POINTER(P), c_int, c_int]
            lib.hipblasLtMatmulDescSetAttribute.argtypes = [P, c_int, P, c_size_t]
            lib.hipblasLtMatrixLayoutCreate.argtypes = [POINTER(P), c_int, c_uint64, c_uint64, c_int64]
            lib.hipblasLtMatmulPreferenceCreate.argtypes = [POINTER(P)]
            lib.hipblasLtMatmulPreferenceSetAttribute.argtypes = [P, c_int, P, c_size_t]
            lib.hipblasLtMatmulPreferenceDestroy.argtypes = [P]
            lib.hipblasLtMatmulAlgoGetHeuristic.argtypes = [P, P, P, P, P, P, P, c_int, POINTER(_Heuristic),
                                                            POINTER(c_int)]
            lib.hipblasLtMatmul.argtypes = [P, P, P, P, P, P, P, P, P, P, P, P, POINTER(_Algo), P, c_size_t, P]
            _lib = lib
            break
    return _lib


def available() -> bool:
    return _load() is not None and ctypes.sizeof(_Heuristic) == 56


def require() -> None:
    if not available():
        raise RuntimeError("hipBLASLt cannot be loaded (looked beside torch's libraries and in /opt/rocm/lib): the "
                           "bfloat16 products of more than 32 rows have no other library")


def _ok(status: int, what: str) -> None:
    if status != 0:
        raise RuntimeError(f"hipBLASLt {what} failed with status {status}")


class _Tile:
    """A shape of the tile kernel, among the library's algorithms."""
    __slots__ = ("shape",)

    def __init__(self, shape: int):
        self.shape = shape

    def name(self) -> list:
        return list(tiles.shapes()[self.shape][:2])


def _tile_named(name, k, gated) -> _Tile | None:
    for i, s in enumerate(tiles.shapes()):
        if list(s[:2]) == name and k >= s[2] and (s[3] or not gated):
            return _Tile(i)
    return None


class _Plan:
    """Descriptors of one problem shape and what runs it: the best of the library's algorithms, or a _Tile."""
    __slots__ = ("desc", "lw", "la", "lc", "candidates", "algo", "tiles", "tile", "tuned", "index", "times", "asked")

    def __init__(self, handle, m, n, k, lda, ldw, ldc, out_dtype, aligned, accumulate):
        lib = _lib
        P = c_void_p
        self.desc, self.lw, self.la, self.lc = P(), P(), P(), P()
        _ok(lib.hipblasLtMatmulDescCreate(byref(self.desc), _COMPUTE_32F, _HIP_R_32F), "descriptor")
        for attr, op in ((_DESC_TRANSA, _OP_T), (_DESC_TRANSB, _OP_N)):
            v = c_int32(op)
            _ok(lib.hipblasLtMatmulDescSetAttribute(self.desc, attr, byref(v), 4), "descriptor attribute")
        ctype = _HIP_R_32F if out_dtype == torch.float32 else _HIP_R_16BF
        _ok(lib.hipblasLtMatrixLayoutCreate(byref(self.lw), _HIP_R_16BF, k, n, ldw), "layout")
        _ok(lib.hipblasLtMatrixLayoutCreate(byref(self.la), _HIP_R_16BF, k, m, lda), "layout")
        _ok(lib.hipblasLtMatrixLayoutCreate(byref(self.lc), ctype, n, m, ldc), "layout")
        pref = P()
        _ok(lib.hipblasLtMatmulPreferenceCreate(byref(pref)), "preference")
        ws = c_uint64(WORKSPACE_BYTES)
        _ok(lib.hipblasLtMatmulPreferenceSetAttribute(pref, _PREF_MAX_WORKSPACE, byref(ws), 8), "preference attribute")
        res = (_Heuristic * CANDIDATES)()
        got = c_int(0)
        _ok(lib.hipblasLtMatmulAlgoGetHeuristic(handle, self.desc, self.lw, self.la, self.lc, self.lc, pref, CANDIDATES,
                                                res, byref(got)), "heuristic")
        lib.hipblasLtMatmulPreferenceDestroy(pref)
        self.candidates = [res[i].algo for i in range(got.value)
                           if res[i].state == 0 and res[i].workspace_size <= WORKSPACE_BYTES]
        if not self.candidates:
            raise RuntimeError(f"hipBLASLt has no kernel for a {m} x {n} x {k} bf16 product")
        self.algo, self.index, self.times = self.candidates[0], 0, None
        fits = aligned and (out_dtype == torch.bfloat16 or not accumulate) and tiles.supports(m, n, k, lda, ldw, ldc)
        self.tiles = [_Tile(i) for i in tiles.candidates(m, n, k)] if fits else []
        self.tile = None     # the one of them that runs it, instead of `algo`
        self.tuned = False   # True once the choice was measured here or taken from the plan file
        self.asked = False   # True once the plan file was asked about this shape


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)   # the handle alone: building a Stream object costs 4 us a call


def _run(handle, plan, algo, a, w, out, workspace, beta=_zero, rows=None) -> None:
    """out = a . w^T + beta * out (the library reads and writes the same matrix); rows: those that hold anything."""
    if isinstance(algo, _Tile):      # (a _Tile in place of the library's algorithm)
        ops.gemm_tile(a, w, out, rows, algo.shape, add=beta is not _zero)
        return
    stream = _raw_stream(a.device.index) if _raw_stream is not None else torch.cuda.current_stream(a.device).cuda_stream
    _ok(_lib.hipblasLtMatmul(handle, plan.desc, byref(_one), w.data_ptr(), plan.lw, a.data_ptr(), plan.la, byref(beta),
                             out.data_ptr(), plan.lc, out.data_ptr(), plan.lc, byref(algo), workspace.data_ptr(),
                             WORKSPACE_BYTES, stream), "matmul")


def _flush_buffer(dev) -> torch.Tensor:
    flush = _flush.get(dev)
    if flush is None:
        flush = _flush[dev] = torch.zeros(FLUSH_BYTES // 4, dtype=torch.float32, device=dev)   # summed as it is: no widened copy
    return flush


def flush_caches(dev) -> None:
    """Reads FLUSH_BYTES of other memory, so that what runs next finds its operands in HBM, as a weight is found
    in a model whose other layers have passed through the caches since. Read, not written: lines written here
    would still be on their way out while the timed kernel runs, and compete with it."""
    _flush_buffer(dev).sum()


def _least_of_three(a, m, run) -> float:
    """Milliseconds of run(), each time behind a read that empties the caches and one of the activations a[:m], which in a model were
    written just before (without it 4,096 x 8,192 x 2,048 takes the library 87 and the tile kernel 125 us, in a step both 100); inf where it
    raises."""
    t = float("inf")
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    try:
        run()   # first use of a kernel loads it
        for _ in range(3):   # the least of three: a single timing wanders by a few per cent, as much as the candidates differ
            flush_caches(a.device)
            a[:m].sum()     # (the rows of this product alone: a is a buffer of the engine's largest step)
            start.record()
            run()
            end.record()
            end.synchronize()
            t = min(t, start.elapsed_time(end))
    except RuntimeError:
        t = float("inf")
    return t


def _first_near(times, tie=TIE) -> int:
    """The first within `tie` of the fastest: two measurements a per cent apart choose the same one."""
    fastest = min(times)
    return next(i for i, t in enumerate(times) if t <= fastest * (1.0 + tie)) if fastest < float("inf") else 0


def _in_trains(w, forms, alone) -> list:
    """Milliseconds a launch of each form(weight) in trains with copies of w in turn; alone: what a launch takes about. Nothing waits in
    between, so the chip stays as busy as a step keeps it."""
    room = _flush_buffer(w.device).view(w.dtype)
    n, k = w.shape
    step = -(-((n - 1) * w.stride(0) + k) // 64) * 64       # elements between copies, whole lines
    copies = [w]
    for i in range(min(FLUSH_BYTES // (2 * step), 63)):
        copies.append(room.as_strided((n, k), (w.stride(0), 1), i * step))
        copies[-1].copy_(w)
    launches = [max(4, min(128, round(TRAIN_MS / t))) for t in alone]
    marks, at = [[] for _ in forms], 0
    for _ in range(TRAINS):
        for form, count, mine in zip(forms, launches, marks):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            for i in range(2 * count):
                if i == count:
                    start.record()
                form(copies[at % len(copies)])
                at += 1
            end.record()
            mine.append((start, end))
    torch.cuda.synchronize(w.device)
    return [min(start.elapsed_time(end) for start, end in mine) / count for mine, count in zip(marks, launches)]


def _tune(handle, plan, m, a, w, out, workspace, beta=_zero) -> None:
    """Times every candidate on the call's own operands and keeps the fastest. In a model the weight of a
    product comes from HBM (the layers before have pushed it out of every cache), so each timed run follows a
    read of FLUSH_BYTES of other memory that empties the memory-side cache; timed on a weight that stays cached, kernels win
    that lose in place. A product that adds to its output is timed on a copy of it."""
    if beta is not _zero:
        out = out.clone()
    found = [*plan.candidates, *plan.tiles]
    times = [_least_of_three(a, m, lambda: _run(handle, plan, algo, a, w, out, workspace, beta, m)) for algo in found]
    library = len(plan.candidates)
    plan.index, plan.tuned = _first_near(times[:library]), True
    plan.algo, first = plan.candidates[plan.index], _first_near(times)
    plan.tile = found[first] if first >= library else None
    plan.times = [round(t * 1e3, 1) if t < float("inf") else None for t in times]
    if _settings["log"]:
        print(f"[dinfer_amd] product {m} x {tuple(out.shape)[1]} x {tuple(a.shape)[1]}, {out.dtype}: algorithm {first} of "
              f"{plan.times} (us)", file=sys.stderr, flush=True)


def _shape_key(m, n, k, lda, ldw, ldc, out_dtype, aligned, accumulate) -> str:
    return f"{m},{n},{k},{lda},{ldw},{ldc},{'f32' if out_dtype == torch.float32 else 'bf16'},{int(accumulate)}{'' if aligned else ',odd'}"


def chosen() -> list:
    """What every shape met so far runs with: rows, columns, depth, index in the library's list (None: "tile", the rows and columns of
    the tile kernel that runs it instead), how it was chosen. Products that a tile runs together with what follows them are named by their "end"."""
    out = []
    for key, plan in _plans.items():
        if plan:
            _, m, n, k = key[:4]
            out.append({"m": m, "n": n, "k": k, "accumulate": bool(key[-1]), "algorithm": plan.index if plan.tile is None else None,
                        "chosen": "measured" if plan.tuned else "first suggestion"})
            if plan.tile is not None:
                out[-1]["tile"] = plan.tile.name()
    for (_, m, n, k, *_, end), plan in _ends.items():
        if plan.tile is not None:
            out.append({"m": m, "n": n, "k": k, "accumulate": False, "algorithm": None, "chosen": "measured", "tile": plan.tile.name(), "end": end})
    return out


def matmul(a: torch.Tensor, w: torch.Tensor, out: torch.Tensor, m: int, accumulate: bool = False, rows: int | None = None) -> bool:
    """out[:m] = a[:m] @ w.T; a, w bfloat16 with contiguous rows, out bfloat16 or float32. accumulate: out[:m] +=
    instead, the sum of the float accumulators and out rounded once. rows: those of the m that hold anything (the shape
    is chosen by m; the tile kernel leaves the others). False, and nothing done, where the library has no algorithm for the shape."""
    require()
    if not (a.stride(1) == 1 and w.stride(1) == 1 and out.stride(1) == 1):
        raise ValueError("library products take operands with contiguous rows")
    beta = _one if accumulate else _zero
    dev = a.device
    handle = _handles.get(dev)
    if handle is None:
        handle = c_void_p()
        with torch.cuda.device(dev):
            _ok(_lib.hipblasLtCreate(byref(handle)), "create")
            _workspaces[dev] = torch.empty(WORKSPACE_BYTES, dtype=torch.uint8, device=dev)
        _handles[dev] = handle
    n, k = w.shape
    aligned = (a.data_ptr() | w.data_ptr() | out.data_ptr()) % 16 == 0      # (the tile kernel asks for it)
    key = (dev, m, n, k, a.stride(0), w.stride(0), out.stride(0), out.dtype, aligned, accumulate)
    plan = _plans.get(key)
    if plan is None:
        try:
            plan = _Plan(handle, m, n, k, a.stride(0), w.stride(0), out.stride(0), out.dtype, aligned, accumulate)
        except RuntimeError:
            plan = False   # a shape the library takes no algorithm for
        _plans[key] = plan
    if plan is False:
        return False
    workspace = _workspaces[dev]
    if (not plan.tuned and _settings["tuning"] == "measured" and m >= TUNE_FROM_ROWS and m * n * k >= TUNE_FROM_WORK
            and len(plan.candidates) > 1):
        _choose(handle, plan, key, a, w, out, workspace, beta)
    _run(handle, plan, plan.algo if plan.tile is None else plan.tile, a, w, out, workspace, beta, m if rows is None else rows)
    return True


def _choose(handle, plan, key, a, w, out, workspace, beta) -> None:
    """Gives a shape its algorithm: from the plan file if it is there (and names a candidate the library still
    lists at that place), else, inside measuring(), by timing. Outside measuring() a shape without a stored choice
    keeps the library's first suggestion and stays open for a later warm-up."""
    global _stored_dirty, worth_measuring_met
    worth_measuring_met += 1
    if plan.asked and not _measuring:
        return
    dev = key[0]
    skey = _shape_key(*key[1:])
    stored = _load_stored(dev)
    known = None if plan.asked else stored.get(skey)
    plan.asked = True
    if isinstance(known, dict):
        i, tile = known.get("index", -1), known.get("tile")
        if 0 <= i < len(plan.candidates) and bytes(plan.candidates[i].data).hex() == known.get("algo"):
            own = next((t for t in plan.tiles if t.name() == tile), None)
            if tile is None or own is not None:
                plan.algo, plan.tile, plan.index, plan.tuned = plan.candidates[i], own, i, True
                return
    if not _measuring or torch.cuda.is_current_stream_capturing():
        return
    _tune(handle, plan, key[1], a, w, out, workspace, beta)
    stored[skey] = {"index": plan.index, "algo": bytes(plan.algo.data).hex()}
    if plan.tile is not None:
        stored[skey]["tile"] = plan.tile.name()
    _stored_dirty = True


class _End:
    """What runs a product with what follows it: a _Tile, or None (the product and a pass of its own)."""
    __slots__ = ("tile", "tuned", "asked", "times")

    def __init__(self):
        self.tile, self.tuned, self.asked, self.times = None, False, False, None


_ends: dict = {}


def with_end(a: torch.Tensor, w: torch.Tensor, out: torch.Tensor, m: int, end: str, rows: int,
             separate: Callable[[torch.Tensor], None]) -> bool:
    """out[:rows] = end(a @ w.T) in one kernel, bfloat16: end "gated" (w = [wg; wu] stacked, silu(a @ wg.T) * (a @ wu.T)) or an
    activation of ops.GEMM_TILE_ACTS. m: the row count the choice goes by; while measuring, out's rows up to m are written. False, and nothing
    done, where `separate`, which does the same with the weight it is given by a product and a pass of its own, was measured to be as
    fast (TRAIN_TIE), or nothing was measured."""
    global _stored_dirty, worth_measuring_met
    gated = end == "gated"
    n, k = w.shape
    if (_settings["tuning"] != "measured" or m < TUNE_FROM_ROWS or m * n * k < TUNE_FROM_WORK or not out.dtype == a.dtype == torch.bfloat16
            or not (a.stride(1) == 1 and w.stride(1) == 1 and out.stride(1) == 1) or (a.data_ptr() | w.data_ptr() | out.data_ptr()) % 16):
        return False
    shape = (m, n, k, a.stride(0), w.stride(0), out.stride(0), end)
    plan = _ends.get((a.device, *shape))
    if plan is None:
        plan = _ends[(a.device, *shape)] = _End()
        plan.tuned = not tiles.supports(*shape[:-1], gated=gated)
    if not plan.tuned:
        worth_measuring_met += 1
        _choose_end(plan, shape, a, w, out, separate, gated)
    if plan.tile is None:
        return False
    ops.gemm_tile(a, w, out, rows, plan.tile.shape, gated=gated, act=None if gated else end)
    return True


def _choose_end(plan, shape, a, w, out, separate, gated) -> None:
    """As _choose, for with_end."""
    global _stored_dirty
    if plan.asked and not _measuring:
        return
    skey = ",".join(map(str, shape))
    stored = _load_stored(a.device)
    known = None if plan.asked else stored.get(skey)
    plan.asked = True
    if isinstance(known, dict) and "tile" in known:
        name = known["tile"]
        plan.tile = _tile_named(name, shape[2], gated) if name is not None else None
        plan.tuned = name is None or plan.tile is not None
        if plan.tuned:
            return
    if not _measuring or torch.cuda.is_current_stream_capturing():
        return
    m, n, k = shape[:3]
    found = [_Tile(i) for i in tiles.candidates(m, n, k, gated)]
    end = shape[-1]
    forms = [separate, *(lambda weight, t=t: ops.gemm_tile(a, weight, out, m, t.shape, gated=gated, act=None if gated else end) for t in found)]
    alone = [_least_of_three(a, m, lambda: form(w)) for form in forms]
    plan.tuned = True
    if min(alone) == float("inf"):
        return      # nothing could be timed: a pass of its own, and no choice in the file
    near = sorted(alone[1:])[:TRAIN_TILES]
    tried = [i for i, t in enumerate(alone) if t < min(alone) * TRAIN_CLEAR and (i == 0 or (t <= near[-1] and t <= near[0] * 1.05))]
    trains = _in_trains(w, [forms[i] for i in tried], [alone[i] for i in tried]) if len(tried) > 1 else [alone[tried[0]]]
    best = tried[_first_near(trains, TRAIN_TIE)]
    plan.tile = found[best - 1] if best else None
    plan.times = [round(t * 1e3, 1) if t < float("inf") else None for t in alone], {i: round(t * 1e3, 1) for i, t in zip(tried, trains)}
    if _settings["log"]:
        print(f"[dinfer_amd] product {m} x {n} x {k} and {end}: {plan.tile.name() if plan.tile else 'a pass of its own'} of {plan.times} (us)",
              file=sys.stderr, flush=True)
    stored[skey] = {"tile": plan.tile.name() if plan.tile else None}
    _stored_dirty = True
