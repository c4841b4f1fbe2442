"""Launch-shape autotuner for the fused DP kernels.

The fused forward and backward kernels (csrc/dp_fused.hip) run a persistent
grid, one atom per wavefront, unless short neighbor buckets put several atoms
on one (dp_fused.short_buckets), where no shape is set. Four launch choices
change their speed but not their results:
  * the wavefronts per block (2, 4 or 8 atoms sharing one block's staged
    weights and LDS; each is a separate instantiation of the kernels);
  * the grid's block cap (how many blocks stride over the atoms);
  * whether the weights of every type pair are staged in LDS per block or read
    through the caches from global memory (LDS costs occupancy as T grows);
  * the XCD-aware block order, which gives each of the eight XCDs (and its L2)
    one contiguous range of atoms instead of every eighth block.
``tune_fused`` times each candidate on the caller's own workload (coordinate
descent: the forward kernel's shape, then the backward's), keeps the fastest,
sets it in the library (matpl_dp_fused_set_launch, process-wide) and caches it
in a JSON file keyed by device, library build (content hash), net width, types,
list width, atom count (rounded to a power of two) and precision. A later call with the same key
reuses the cached shape without timing.
"""
from __future__ import annotations

import hashlib
import json
import math
import os
from typing import Callable, Dict, Optional

import torch

from . import _lib

BLOCK_CAPS = (512, 768, 1024, 1536, 2048, 3072, 4096, 8192, 16384)
WAVES = (2, 4, 8)
# the shape that leaves the choice to the library (by size, types and precision, groups of atoms included)
DEFAULT = {"max_blocks": 4096, "lds_weights": -1, "xcd": 0, "waves": 4}


def set_launch(kernel: int, max_blocks: int, lds_weights: int, xcd: int, waves: int = 4) -> None:
    _lib.call("matpl_dp_fused_set_launch", kernel, max_blocks, lds_weights, xcd)
    _lib.call("matpl_dp_fused_set_waves", kernel, waves)


def reset() -> None:
    for k in (0, 1):
        set_launch(k, **DEFAULT)


def cache_path() -> str:
    return os.environ.get("MATPL_TUNE_CACHE",
                          os.path.join(os.path.expanduser("~"), ".cache", "matpl_amd", "fused_launch.json"))


def device_id() -> str:
    """GPU architecture and CU count (the marketing name can read empty under a profiler)."""
    if not torch.cuda.is_available():
        return "cpu"
    p = torch.cuda.get_device_properties(torch.cuda.current_device())
    arch = getattr(p, "gcnArchName", "") or p.name or "gpu"
    return f"{arch.split(':')[0]}x{p.multi_processor_count}"


def parse_launch(spec: str) -> Dict:
    """'fb,fl,fx,bb,bl,bx' (blocks, LDS weights, XCD order of the forward, then the backward kernel;
    4 wavefronts per block) or 'fb,fl,fx,fw,bb,bl,bx,bw' (with the wavefronts per block)."""
    v = [int(x) for x in spec.split(",")]
    if len(v) == 6:
        v = v[:3] + [4] + v[3:] + [4]
    if len(v) != 8:
        raise ValueError("launch spec needs 6 or 8 integers: fwd blocks,lds,xcd[,waves],bwd blocks,lds,xcd[,waves]")
    f = {"max_blocks": v[0], "lds_weights": v[1], "xcd": v[2], "waves": v[3]}
    b = {"max_blocks": v[4], "lds_weights": v[5], "xcd": v[6], "waves": v[7]}
    set_launch(0, **f)
    set_launch(1, **b)
    return {"forward": f, "backward": b, "fixed": True}


_BUILD_ID = None


def build_id() -> str:
    """Content hash of the loaded libmatpl_hip.so: a shape tuned for one build of the fused kernels
    is not reused for another."""
    global _BUILD_ID
    if _BUILD_ID is None:
        h = hashlib.sha1()
        with open(_lib.LIB_PATH, "rb") as f:
            for chunk in iter(lambda: f.read(1 << 20), b""):
                h.update(chunk)
        _BUILD_ID = h.hexdigest()[:12]
    return _BUILD_ID


def workload_key(E: int, T: int, mnl: int, m: int, natoms: int, precision: str) -> str:
    dev = device_id()
    nb = 1 << max(0, int(round(math.log2(max(natoms, 1)))))
    return f"{dev}|lib{build_id()}|E{E}|T{T}|mnl{mnl}|m{m}|n~{nb}|{precision}"


def _load() -> Dict:
    try:
        with open(cache_path()) as f:
            return json.load(f)
    except (OSError, ValueError):
        return {}


def _store(key: str, val: Dict) -> None:
    data = _load()
    data[key] = val
    path = cache_path()
    try:
        os.makedirs(os.path.dirname(path), exist_ok=True)
        tmp = path + f".{os.getpid()}"
        with open(tmp, "w") as f:
            json.dump(data, f, indent=1, sort_keys=True)
        os.replace(tmp, path)
    except OSError:
        pass          # an unwritable cache only costs a re-tune next time


def _time(run: Callable[[], None], reps: int) -> float:
    run()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        run()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / reps


def tune_fused(run: Callable[[], None], key: str, reps: int = 10, use_cache: bool = True,
               log: Optional[Callable[[str], None]] = None) -> Dict:
    """Chooses and sets the launch shape of both fused kernels for the workload ``run`` enqueues
    (one whole evaluation on the current stream). Returns {"forward": cfg, "backward": cfg,
    "ms": time per evaluation with the chosen shapes, "ms_default": with the defaults, "cached": bool}."""
    if use_cache:
        hit = _load().get(key)
        if hit:
            for k, name in ((0, "forward"), (1, "backward")):
                set_launch(k, **hit[name])
            return dict(hit, cached=True)
    reset()
    ms_default = _time(run, reps)
    best = {0: dict(DEFAULT), 1: dict(DEFAULT)}
    best_ms = ms_default
    for k in (0, 1):
        for waves in WAVES:
            for lw in (-1, 0):
                for xcd in (0, 1):
                    for cap in BLOCK_CAPS:
                        cand = {"max_blocks": cap, "lds_weights": lw, "xcd": xcd, "waves": waves}
                        if cand == best[k]:
                            continue
                        set_launch(k, **cand)
                        try:
                            ms = _time(run, reps)
                        except _lib.MatplError:
                            continue      # e.g. 8 waves' neighbor tiles exceed the LDS budget
                        if ms < best_ms:
                            best_ms, best[k] = ms, cand
        set_launch(k, **best[k])
    # a fresh measurement of the chosen pair (the search's own minimum is biased low)
    best_ms = _time(run, reps)
    res = {"forward": best[0], "backward": best[1], "ms": round(best_ms, 4), "ms_default": round(ms_default, 4)}
    if log:
        log(f"autotune {key}: {res}")
    _store(key, res)
    return dict(res, cached=False)
