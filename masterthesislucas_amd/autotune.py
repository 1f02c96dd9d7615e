"""Timing of the traversal's settings on a caller's context.

One walk serves every variant id and either issue priority (bh_set_traverse_variant,
bh_set_walk_priority in include/bh.h), and the library chooses the waves per sink group
(bh_set_traverse_split) from the launch size, so a program need not tune. These calls time the
walk on the caller's own context (already holding the workload) with the library's HIP-event
phase timers; `tune_split` selects the fastest number of waves per group. `tune` can remember its
time per (kernel, tree mode, log2 N, theta) in a JSON table next to this file.
"""
from __future__ import annotations

import json
import math
import os

HERE = os.path.dirname(os.path.abspath(__file__))
TABLE = os.path.join(HERE, "tuned_variants.json")

# Points up to which bh_forces with the t-SNE kernel and split 1 takes its own walk (kPreorderMax)
PREORDER_MAX = 131072


def _key(ctx, theta):
    return f"{ctx.kernel}|{ctx.tree_mode}|n{int(math.log2(max(ctx.n, 1)))}|t{theta:.3f}"


def load_table(path=TABLE):
    if os.path.exists(path):
        with open(path) as f:
            return json.load(f)
    return {}


def lookup(ctx, theta, path=TABLE):
    return load_table(path).get(_key(ctx, theta))


def time_variant(ctx, variant, theta, repeats=3):
    """Average traversal milliseconds on the current tree, with variant id `variant` selected."""
    ctx.set_variant(variant)
    ctx.forces_device_only(theta)  # warm the code object and caches
    ctx.profile_enable(True)
    ctx.profile_read(reset=True)
    for _ in range(repeats):
        ctx.forces_device_only(theta)
    ms, launches = ctx.profile_read(reset=True)["traversal"]
    ctx.profile_enable(False)
    return ms / max(launches, 1)


def tune(ctx, theta, repeats=3, save=False, path=TABLE):
    """Time the walk on ctx's current tree (ctx must have been built) and return
    (variant, {variant: ms}). Every variant id and either priority runs the same walk: the
    context keeps the ones it has, and one timing stands for all."""
    best = ctx.variant
    times = {best: time_variant(ctx, best, theta, repeats)}
    if save:
        table = load_table(path)
        table[_key(ctx, theta)] = {"variant": best, "priority": ctx.priority,
                                   "ms": {str(k): v for k, v in times.items()}}
        with open(path, "w") as f:
            json.dump(table, f, indent=1, sort_keys=True)
    return best, times


def split_candidates(ctx, splits):
    """The settings among `splits` that differ for ctx: 3 to 8 ask for four waves alike, and with
    the t-SNE kernel on up to PREORDER_MAX points split 1 is left out where others are offered:
    bh_forces, which these calls time, then takes a walk of its own, while the descent
    (bh_tsne_run) at split 1 takes two or four waves of the common walk, by size."""
    out, seen = [], set()
    for s in splits:
        waves = s if s < 3 else 4
        if waves not in seen:
            seen.add(waves)
            out.append(s)
    if ctx.kernel == "tsne" and ctx.n <= PREORDER_MAX and len(out) > 1:
        out = [s for s in out if s != 1]
    return out


def tune_split(ctx, theta, splits=(1, 2, 4, 8), variants=None, repeats=3):
    """Time the settings `splits` (split_candidates) on ctx's current tree, select the fastest and
    return ((variant, split), {"variant/split": ms}). One variant stands for all unless
    `variants` are given."""
    variants = (ctx.variant,) if variants is None else variants
    times = {}
    for s in split_candidates(ctx, splits):
        ctx.set_split(s)
        for v in variants:
            times[(v, s)] = time_variant(ctx, v, theta, repeats)
    best = min(times, key=times.get)
    ctx.set_variant(best[0])
    ctx.set_split(best[1])
    return best, {f"{v}/{s}": ms for (v, s), ms in times.items()}
