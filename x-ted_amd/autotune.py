"""Autotuner for the granularity cut-overs and the batch schedule.

The reference fixes its granularity thresholds at 15 / 18,750 / 25,250,000
cells (X-TED_GPU/parallel_X_TED.cu:382) from a cost model fitted to one GPU
(supplement, section 2). Here the class rule has knobs (include/xted.h,
xted_set_tuning / xted_set_tail_rule / xted_set_level_align /
xted_set_size_bands / xted_set_light_lds / xted_set_tiny_forms): slot bytes per wave before a
table gets more waves, the most columns per lane, a latency rule for the last levels, where each
pair's levels sit in the batch, the order of a launch's tables and the widest tables the tiny
forms take. This
module times a workload under a staged grid of rules on the device it runs
on:

  1. the schedule: level alignment x size bands (none, by rows, by rows and
     light / heavy slot storage);
  2. the tail rule;
  3. a coarse grid of size bands x slot bytes per wave x columns per lane x
     tiny forms (16 lanes; 16 and 32);
  4. the slot bytes per wave above which a table is heavy (size bands 2);
  5. the tiny forms (tables of up to 16, 32 or 64 columns);
  6. a fine grid of slot bytes per wave (1 KiB steps) around the best;
  7. a confirmation: the best rule and the three next fastest candidates
     re-timed in two interleaved rounds on the tuning workload and on a
     second one (seed stream 1005), the lowest mean of the two median steps
     winning.

The workload is the 4096-pair uneven batch's generator on a seed stream of
its own (not the one bench.py times). The rule starts as a new context's; a
candidate replaces the current best only when every one of its steps is
faster than the best rule's fastest step, so step-to-step noise cannot pick
a rule. Every candidate must reproduce the first rule's distances
exactly, or the run stops.

    python x-ted_amd/autotune.py [--pairs N] [--out x-ted_amd/tuning.json]
"""
import argparse
import itertools
import json
import os
import sys
import time

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)
import xted  # noqa: E402

# A new context's rule (kDefaultRule and the constants after it in csrc/device.hpp).
DEFAULT = {"lds_per_wave": 10 * 1024, "max_cpl": 16, "min_waves": 1, "wide_cols": 1 << 30,
           "tail_pairs": 32, "level_align": 1, "size_bands": 1, "light_lds": 10 * 1024,
           "tiny_forms": 1}
# Where a search starts that names no rule: narrow lanes, every pair from level 0.
START = dict(DEFAULT, max_cpl=8, level_align=0)
# Seed stream of the tuning workload (bench.py times stream 3).
SEED_TUNE = 1003
SEED_CONFIRM = 1005  # second workload of the confirmation round
COARSE_LDS = [6 * 1024, 10 * 1024, 14 * 1024, 20 * 1024, 28 * 1024]
STAGES = [
    {"level_align": [0, 1, 2], "size_bands": [0, 1, 2]},
    {"tail_pairs": [0, 8, 32]},
    # Slot bytes per wave set which tables share a launch, and with it how
    # far splitting light from heavy tables raises occupancy: searched together.
    # The 32-lane tiny form pays only with some of these rules, so it is
    # searched with them too.
    {"size_bands": [1, 2], "lds_per_wave": COARSE_LDS, "max_cpl": [8, 16], "tiny_forms": [1, 3]},
    # Where heavy tables start (size-band mode 2 only).
    {"light_lds": [6 * 1024, 8 * 1024, 10 * 1024, 12 * 1024, 14 * 1024]},
    # Which tables the tiny forms take (16-lane only, up to 32 or 64 columns).
    {"tiny_forms": [1, 3, 7]},
]
FINE_STEP = 1024
FINE_SPAN = 3  # steps either side of the coarse best
# Confirmation: the best rule and the next fastest candidates re-timed in
# interleaved rounds (their best single steps are within noise of each other).
CONFIRM_TOP = 4
CONFIRM_ROUNDS = 2
TUNING_FILE = os.path.join(HERE, "tuning.json")


def apply(ctx, rule):
    ctx.set_tuning(rule["lds_per_wave"], rule["max_cpl"], rule["min_waves"], rule["wide_cols"])
    ctx.set_tail_rule(rule["tail_pairs"])
    ctx.set_level_align(rule["level_align"])
    ctx.set_size_bands(rule["size_bands"])
    ctx.set_light_lds(rule["light_lds"])
    ctx.set_tiny_forms(rule["tiny_forms"])


def load(path=TUNING_FILE):
    """The stored rule, or the default when none was stored."""
    try:
        with open(path) as f:
            rule = json.load(f)["rule"]
        return {k: int(rule.get(k, DEFAULT[k])) for k in DEFAULT}
    except (OSError, KeyError, ValueError):
        return dict(DEFAULT)


def steps(ctx, xs, ys, rule, reps):
    """Per-step times of `reps` batches under `rule` (after a warm-up) and
    the distances."""
    apply(ctx, rule)
    dist, _, _ = ctx.batch(xs, ys)  # warm (plans, captures the graph)
    times = []
    for _ in range(reps):
        t = time.perf_counter()
        d, _, _ = ctx.batch(xs, ys)
        times.append(time.perf_counter() - t)
        if not np.array_equal(d, dist):
            raise RuntimeError("distances changed between runs")
    return times, dist


def tune(ctx, xs, ys, stages=STAGES, reps=3, log=print, confirm_top=CONFIRM_TOP, confirmed=None,
         confirm_sets=(), start=None):
    """Returns (best_rule, results, spread): the staged search described in
    the module docstring, from the rule start (START). results lists (rule, best step time); confirmed, if
    given, receives (rule, score) of the confirmation round, the score being
    the mean over (xs, ys) and the workloads of confirm_sets (pairs of id
    arrays) of each one's median step time."""
    base = dict(START if start is None else start)
    base_times, base_d = steps(ctx, xs, ys, base, 6)
    spread = max(base_times) - min(base_times)
    base_t = min(base_times)
    results = [(dict(base), base_t)]
    log(f"start {base}: {base_t * 1e3:.1f} ms, step-to-step spread {spread * 1e3:.2f} ms")
    # The best rule's fastest step: a candidate wins only when its slowest
    # step beats it (every step of the candidate faster than every step of
    # the best), so neither rule's step-to-step noise can pick it.
    best, best_t = dict(base), base_t

    def trial(rule):
        nonlocal best, best_t
        if any(rule == r for r, _ in results):
            return
        try:
            times, d = steps(ctx, xs, ys, rule, reps)
        except xted.XtedError as e:
            log(f"{rule}: rejected ({e})")
            return
        if not np.array_equal(d, base_d):
            raise RuntimeError(f"rule {rule} changed a distance")
        t = min(times)
        results.append((rule, t))
        won = max(times) < best_t
        log(f"{rule}: {t * 1e3:.1f} ms (slowest step {max(times) * 1e3:.1f})"
            f"{' (new best)' if won else ''}")
        if won:
            best, best_t = rule, t

    for grid in stages:
        keys = list(grid)
        around = dict(best)
        for vals in itertools.product(*(grid[k] for k in keys)):
            trial(dict(around, **dict(zip(keys, vals))))
    # Fine steps of slot bytes per wave around the coarse best.
    around = dict(best)
    for k in range(-FINE_SPAN, FINE_SPAN + 1):
        lds = around["lds_per_wave"] + k * FINE_STEP
        if lds >= 2 * 1024:
            trial(dict(around, lds_per_wave=lds))
    # Confirmation: the best rule and the fastest other candidates (by their
    # best step), re-timed in interleaved rounds; the lowest median step wins.
    ranked = [r for r, _ in sorted(results, key=lambda rt: rt[1]) if r != best]
    finalists = [best] + ranked[:max(0, confirm_top - 1)]
    sets = [(xs, ys, base_d)]
    for cx, cy in confirm_sets:
        sets.append((cx, cy, steps(ctx, cx, cy, base, 1)[1]))
    samples = [[[] for _ in sets] for _ in finalists]
    if len(finalists) > 1:
        for _ in range(CONFIRM_ROUNDS):
            for i, rule in enumerate(finalists):
                for w, (sx, sy, sd) in enumerate(sets):
                    times, d = steps(ctx, sx, sy, rule, reps)
                    if not np.array_equal(d, sd):
                        raise RuntimeError(f"rule {rule} changed a distance")
                    samples[i][w].extend(times)
        scores = [float(np.mean([np.median(t) for t in per])) for per in samples]
        for rule, per, sc in zip(finalists, samples, scores):
            meds = ", ".join(f"{np.median(t) * 1e3:.1f}" for t in per)
            log(f"confirm {rule}: medians {meds} ms, mean {sc * 1e3:.1f} ms")
            if confirmed is not None:
                confirmed.append((rule, sc))
        best = finalists[int(np.argmin(scores))]
    apply(ctx, best)
    return best, results, spread


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--pairs", type=int, default=4096)
    ap.add_argument("--out", default=TUNING_FILE)
    args = ap.parse_args()
    sys.path.insert(0, os.path.dirname(HERE))
    from bench import batch_trees
    trees = batch_trees(args.pairs, cfg=SEED_TUNE)
    trees2 = batch_trees(args.pairs, cfg=SEED_CONFIRM)
    confirmed = []
    with xted.Context(0) as ctx:
        ids = ctx.pool_add(trees)
        ids2 = ctx.pool_add(trees2)
        best, results, spread = tune(ctx, ids[0::2].copy(), ids[1::2].copy(),
                                     confirmed=confirmed, start=DEFAULT,
                                     confirm_sets=[(ids2[0::2].copy(), ids2[1::2].copy())])
    out = {"rule": best,
           "workload": f"batch{args.pairs}_uneven_n100-1000_deep50_shallow50_alphabet200 "
                       f"(seed stream {SEED_TUNE})",
           "spread_ms": round(spread * 1e3, 2),
           "results_ms": [{"rule": r, "ms": round(t * 1e3, 2)} for r, t in results],
           "confirm_workload": f"seed stream {SEED_CONFIRM}",
           "confirm_mean_median_ms": [{"rule": r, "ms": round(t * 1e3, 2)} for r, t in confirmed]}
    with open(args.out, "w") as f:
        json.dump(out, f, indent=1)
    print(json.dumps({"best": best, "spread_ms": round(spread * 1e3, 2)}))


if __name__ == "__main__":
    main()
