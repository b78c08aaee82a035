"""The cost tables of choose_plan (fast_infer_amd/csrc/int4_gemm.hip) from their timings.

    python profiles/linear_plans.py            # fit, print the tables and how well they choose
    python profiles/linear_plans.py --held-out # fit on half of the sizes, judge on the others

linear_plan_timings.txt.gz holds 8232 sizes of a linear call, one per line: weight form, rows M,
columns N, depth K, and the time in us of each plan tried, ``m<rows>x<columns>/<K splits>`` for
mid_gemm_kernel, ``d...`` for tile_gemm_kernel (packed weights: with the unpacking pass) and ``g``
for gemv_kernel.  The sizes are random over 1 to 30000 rows, 88 to 28672 columns (odd ones among
them) and K 128 to 14336.  A time is the fastest of seven replays of a HIP graph of four to eight
calls with different weights, on one MI355X, in a build in which the plan could be forced.

The fit is a least-squares fit of the logarithms, plans near the fastest of their size weighted
most.  Needs numpy and scipy.
"""

import collections
import gzip
import math
import random
import sys
from pathlib import Path

import numpy as np
from scipy.optimize import least_squares, nnls

CUS, MAX_SPLITS, DENSE_MIN_M, GEMV_MAX_M = 256, 16, 129, 16
# dense, rows, columns, workgroups per CU, may split K
TILES = {"packed": [(0, 16, 64, 4, 1), (0, 32, 64, 4, 1), (0, 64, 64, 4, 1), (0, 64, 128, 4, 1),
                    (0, 128, 64, 2, 1), (0, 128, 128, 2, 1), (1, 128, 128, 2, 0), (1, 256, 256, 1, 0)],
         "fp16": [(1, 32, 64, 2, 1), (1, 64, 64, 2, 1), (1, 64, 128, 2, 1), (1, 128, 64, 2, 1),
                  (1, 128, 128, 2, 1), (1, 256, 256, 1, 0)]}
GEMV = ("g",)


def ceil_div(a, b):
    return -(-a // b)


def load():
    sizes = {}
    with gzip.open(Path(__file__).with_name("linear_plan_timings.txt.gz"), "rt") as f:
        for line in f:
            form, m, n, k, *plans = line.split()
            times = {}
            for p in plans:
                name, us = p.split("=")
                if name == "g":
                    times[GEMV] = float(us)
                else:
                    tile, splits = name[1:].split("/")
                    mt, nt = tile.split("x")
                    times[(int(name[0] == "d"), int(mt), int(nt), int(splits))] = float(us)
            sizes[(form, int(m), int(n), int(k))] = times
    return sizes


def weight_mb(form, dense, n, k):
    return n * k * (0.5e-6 if form == "packed" and not dense else 2e-6)


def unpacking(form, dense, n, k):
    return 2.5 + 0.62e-6 * n * k if form == "packed" and dense else 0.0


def tile_terms(form, tile, m, n, k, s):
    """What tile_cost adds up: 1, rounds by their load, workgroups on a CU, MB, K split."""
    dense, mt, nt, per_cu, splits = tile
    tiles_n = ceil_div(n, nt)
    on_cu = ceil_div(s * ceil_div(ceil_div(m, mt) * tiles_n, 8), CUS // 8)
    load = [0.0] * per_cu
    per = ceil_div(k // 128, s)
    load[per_cu - 1] += per * (on_cu // per_cu)
    if on_cu % per_cu:
        load[on_cu % per_cu - 1] += per
    x = [1.0, *load, on_cu - 1, weight_mb(form, dense, n, k)]
    if splits:
        x += [float(s > 1), float(s) if s > 1 else 0.0]
    return x + [tiles_n * m * k * 2e-6]


def gemv_terms(form, m, n, k):
    groups, load = k // 128, ceil_div(ceil_div(n, 16), CUS)
    passes = ceil_div(groups, 24 if form == "packed" else 12) - 1
    return [1.0, load - 1, groups, groups * load * m, weight_mb(form, 0 if form == "packed" else 1, n, k),
            passes, passes * (load - 1), load * m]


def solve(rows):
    x, us, w = (np.array(c, dtype=float) for c in zip(*rows))
    us = np.maximum(us, 1.0)
    scale = np.sqrt(w)
    start, _ = nnls(x * (scale / us)[:, None], scale)
    fit = least_squares(lambda p: (np.log(np.maximum(x @ p, 0.3)) - np.log(us)) * scale,
                        np.maximum(start, 1e-4), loss="soft_l1", f_scale=0.08, bounds=(0, np.inf),
                        x_scale=np.maximum(start, 1e-2))
    return fit.x


def fit(sizes):
    rows = collections.defaultdict(list)
    for (form, m, n, k), times in sizes.items():
        best = min(times.values())
        for plan, us in times.items():
            w = math.exp(-8 * min(us / best - 1, 1.0)) + 0.01
            if plan == GEMV:
                rows[form, GEMV].append((gemv_terms(form, m, n, k), us, w))
                continue
            tile = next(t for t in TILES[form] if t[:3] == plan[:3])
            rows[form, tile].append((tile_terms(form, tile, m, n, k, plan[3]),
                                     us - unpacking(form, tile[0], n, k), w))
    return {key: solve(r) for key, r in rows.items()}


def predict(model, size, plan):
    form, m, n, k = size
    if plan == GEMV:
        return 0.97 * float(np.dot(gemv_terms(*size), model[form, GEMV]))
    tile = next(t for t in TILES[form] if t[:3] == plan[:3])
    us = float(np.dot(tile_terms(form, tile, m, n, k, plan[3]), model[form, tile]))
    x_mb = 2e-6 * m * k
    if x_mb > 32:
        us = max(us, 0.13 * ceil_div(n, tile[2]) * x_mb)
    return us * (0.98 if tile[1] == 256 else 1.0) + unpacking(form, tile[0], n, k)


def allowed(size, plan):
    """Plans that choose_plan weighs."""
    form, m, n, k = size
    if plan == GEMV:
        return m <= GEMV_MAX_M
    dense, mt, nt, s = plan
    tiles = ceil_div(m, mt) * ceil_div(n, nt)
    return (s <= MAX_SPLITS and not (form == "packed" and dense and m < DENSE_MIN_M)
            and not (mt > 32 and mt >= 2 * m) and not (mt < 128 and m > 8 * mt and tiles > 1024)
            and not (s > 1 and (tiles > 2048 or tiles * s > 5 * CUS))
            and not (s > 1 and m >= DENSE_MIN_M
                     and s * ceil_div(m, mt) * mt * ceil_div(n, nt) * nt * 4 > n * k * 2))


def judge(model, sizes):
    lost = []
    for size, times in sizes.items():
        times = {p: us for p, us in times.items() if allowed(size, p)}
        chosen = min(times, key=lambda p: predict(model, size, p))
        lost.append((times[chosen] / min(times.values()), size, chosen))
    lost.sort(reverse=True)
    over = [r[0] for r in lost]
    mean = math.exp(sum(map(math.log, over)) / len(over))
    print(f"{len(over)} sizes: {100 * (mean - 1):.1f}% over the fastest plan timed on average, "
          f"{100 * (np.percentile(over, 95) - 1):.0f}% at the 95th percentile, "
          f"{100 * (over[0] - 1):.0f}% at worst ({lost[0][1]}, {lost[0][2]})")


def number(x, digits=3):
    text = f"{x:.{digits}f}".rstrip("0")
    return text + ("0f" if text.endswith(".") else "f")


def show(model):
    for form, name in (("packed", "kPackedTiles"), ("fp16", "kHalfTiles")):
        print(f"constexpr TileCost {name}[] = {{")
        for tile in TILES[form]:
            dense, mt, nt, per_cu, splits = tile
            th = list(model[form, tile])
            load, (wg, mb), x_mb = th[1:1 + per_cu], th[1 + per_cu:3 + per_cu], th[-1]
            split = [number(v) for v in th[3 + per_cu:5 + per_cu]] if splits else ["0", "0"]
            print(f"    {{{'true' if dense else 'false'}, {mt}, {nt}, {per_cu}, {number(th[0])}, "
                  f"{{0, {', '.join(map(number, load))}}}, {', '.join(split)}, {number(wg)}, "
                  f"{number(mb, 4)}, {number(x_mb, 4)}}},")
        print("};")
    for form in TILES:
        print(f"gemv_cost, {form}: 1, load - 1, groups, groups x load x M, MB, passes, "
              f"passes x (load - 1), load x M\n   ", ", ".join(number(v, 4) for v in model[form, GEMV]))


if __name__ == "__main__":
    data = load()
    if "--held-out" in sys.argv:
        keys = sorted(data)
        random.Random(1).shuffle(keys)
        half = len(keys) // 2
        judge(fit({k: data[k] for k in keys[:half]}), {k: data[k] for k in keys[half:]})
    else:
        model = fit(data)
        show(model)
        judge(model, data)
