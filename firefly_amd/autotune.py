"""Autotuner for the launch shapes.

Times renders of the actual request for a few paths-in-flight choices (samples
per pixel in flight, spp_batch).  Renders and uncounted traces take their
traversal shape from the number of rays; the traversal variants (see
ff_traversal_variant_info) shape the traces that count, so those are timed for
the variants.  The variant found is kept on the context.  Results can be written
as JSON and reused.
"""
from __future__ import annotations

import json
import time
from typing import Dict, Iterable, Optional

from . import abi


def _time_render(ctx, scene, env, cam, w, h, spp, depth, seed, film, spp_batch, reps):
    import torch
    best = float("inf")
    for _ in range(reps):
        film.zero_()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        abi.render(ctx, scene, env, cam, w, h, spp, depth, seed, film, spp_batch=spp_batch)
        torch.cuda.synchronize()
        best = min(best, time.perf_counter() - t0)
    return best


def _time_traces(ctx, scene, cam, w, h, seed, variants, reps):
    """Seconds of a counted closest-hit trace of the request's camera rays, for each variant."""
    import torch
    rays = torch.empty((w * h, 8), dtype=torch.float32, device="cuda")
    hits = torch.empty((w * h, 4), dtype=torch.float32, device="cuda")
    counts = torch.zeros(2, dtype=torch.int64, device="cuda")
    abi.generate_rays(ctx, cam, w, h, seed, 0, rays)
    out = []
    for var in variants:
        abi.set_traversal_variant(ctx, var[0])
        scene.trace_closest(rays, hits, counts_dev=counts)  # (code-object load)
        best = float("inf")
        for _ in range(reps):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            scene.trace_closest(rays, hits, counts_dev=counts)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t0)
        out.append(best)
    return out


def autotune(ctx: abi.Context, scene: abi.Scene, env: abi.EnvMap, cam: abi.Camera, width: int, height: int,
             max_depth: int, seed: int = 0, probe_spp: int = 2, batches: Iterable[int] = (1, 2),
             reps: int = 2, out_json: Optional[str] = None, refine_batches: Iterable[int] = (),
             refine_spp: int = 0, tail_candidates: Iterable[int] = (), tail_from: Iterable[int] = (3, 4, 5)) -> Dict:
    """Pick the fastest spp_batch for this request, and the fastest traversal
    variant for traces that count (closest hits of the request's camera rays).

    Without `refine_spp`: `probe_spp` samples per pixel with each spp_batch of
    `batches`.  With `refine_spp` (the request's spp): that many samples with
    each spp_batch of `batches` and `refine_batches` -- more paths in flight mean
    fewer traversal launches, each paying the latency of its slowest ray once.
    All times are the best of `reps`.

    No launch has a second variant for late bounces any more: `tail_candidates`
    and `tail_from` are accepted, and the choice for them is none (-1).  Returns
    a dict with the choice and every timing ("candidates": renders, "traces":
    counted traces)."""
    import torch
    film = torch.zeros((height, width, 4), dtype=torch.float32, device="cuda")
    variants = abi.traversal_variants()
    # warm-up (first launches pay code-object load and allocation)
    abi.render(ctx, scene, env, cam, width, height, 1, max_depth, seed, film)
    torch.cuda.synchronize()

    def entry(var, k, t, spp):
        v, block, lds, refill, ww, width_bvh = var
        return {"variant": v, "block": block, "lds_entries": lds, "refill": refill, "while_while": ww,
                "bvh_width": width_bvh, "spp_batch": k, "seconds": t, "probe_spp": spp}

    seconds = _time_traces(ctx, scene, cam, width, height, seed, variants, reps)
    chosen = variants[min(range(len(variants)), key=seconds.__getitem__)]
    abi.set_traversal_variant(ctx, chosen[0])
    spp = refine_spp if refine_spp > 0 else probe_spp
    ks = sorted(set(list(batches) + (list(refine_batches) if refine_spp > 0 else [])))
    results = []
    for k in (k for k in ks if k <= spp):
        t = _time_render(ctx, scene, env, cam, width, height, spp, max_depth, seed, film, k, reps)
        results.append(entry(chosen, k, t, spp))
    best = min(results, key=lambda r: r["seconds"])
    if refine_spp > 0 and list(tail_candidates):
        best = dict(best, tail_variant=-1, tail_from=0)
    out = {"best": best, "candidates": results,
           "traces": [{"variant": v[0], "seconds": t} for v, t in zip(variants, seconds)],
           "request": {"width": width, "height": height, "max_depth": max_depth, "probe_spp": probe_spp,
                       "refine_spp": refine_spp}}
    if out_json:
        with open(out_json, "w") as f:
            json.dump(out, f, indent=1)
    return out
