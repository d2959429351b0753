"""Tile-shape autotuner of the stencil pass of two-pass plans.

    python -m sympygr_amd.autotune [--sizes 9 13 17 ...] [--top 6] [--dry-run]

For each interior size n it lists the tile shapes (tx, ty, tz) the general
stencil kernel admits (at most 512 points, halo and stage arrays within its
LDS), ranks them by a cost model (points computed per interior point, halo
loads, mixed-derivative stage cells and x-row length per tile point), times
the best few and 8^3 on a uniform tiling of n^3 blocks (one
RHS, mixed precision, upwind; SGR_TILE_SHAPE forces each shape), and keeps the fastest.
It writes the table sgr_plan_create reads (default
sympygr_amd/csrc/gen/tile_table.inc; rebuild the library afterwards) and a
report with every timing (default profiles/tile_autotune.json).  Needs a GPU.
"""
from __future__ import annotations

import argparse
import json
import os
import subprocess
import sys
import time

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
TABLE = os.path.join(PKG, "csrc", "gen", "tile_table.inc")
REPORT = os.path.join(ROOT, "profiles", "tile_autotune.json")

# the general kernel's LDS limits (csrc/bssn_common.h)
TILE_PTS, U_CAP, DX_CAP, DY_CAP = 512, 3456, 3200, 1600


def shape_ok(tx, ty, tz):
    return (min(tx, ty, tz) >= 2 and tx * ty * tz <= TILE_PTS and (tx + 6) * (ty + 6) * (tz + 6) <= U_CAP and
            tx * (ty + 6) * (tz + 6) <= DX_CAP and tx * ty * (tz + 6) <= DY_CAP)


def cost(n, s):
    """Model: points the tiles compute per interior point (idle threads of a
    tile under 512 points counted as work), times the per-point work of a
    tile: halo points loaded, the mixed-derivative stage cells (6/ty + 12/tz
    stencils per point) and short x-rows (partial cache lines in the halo
    loads and workspace stores)."""
    tx, ty, tz = s
    waste = 1.0
    for t in s:
        waste *= -(-n // t) * t / n
    busy = TILE_PTS / (tx * ty * tz)
    halo = (tx + 6) * (ty + 6) * (tz + 6) / (tx * ty * tz)
    stage = 6.0 / ty + 12.0 / tz
    return waste * busy * (1.0 + 0.25 * halo + 0.1 * stage) * (1.0 + 2.0 / tx)


def candidates(n, top):
    c = [(tx, ty, tz) for tx in range(2, n + 1) for ty in range(2, n + 1) for tz in range(2, n + 1)
         if shape_ok(tx, ty, tz)]
    c.sort(key=lambda s: cost(n, s))
    out = [s for s in c[:top]]
    if (8, 8, 8) not in out:
        out.append((8, 8, 8))
    return out


def time_shape(n, shape, steps=10):
    import torch
    import sympygr_amd as sgr
    from sympygr_amd import data
    nb = max(2, round((12e6 / n ** 3) ** (1.0 / 3.0)))
    bl = data.uniform_tiling(nb=nb, n=n, stagger=0.5)
    u = data.fill_blocks(bl, backend="torch", device="cuda")
    out = torch.zeros_like(u)
    os.environ["SGR_TILE_SHAPE"] = ",".join(str(x) for x in shape)
    try:
        plan = sgr.Plan(bl, sgr.params(adv="upwind", precision="mixed", ko_sigma=0.1))
    finally:
        del os.environ["SGR_TILE_SHAPE"]
    for _ in range(2):
        plan.rhs(out, u)
    torch.cuda.synchronize()
    best = float("inf")
    for _ in range(3):
        t0 = time.perf_counter()
        for _ in range(steps):
            plan.rhs(out, u)
        torch.cuda.synchronize()
        best = min(best, (time.perf_counter() - t0) / steps)
    pts = bl.interior_points()
    del plan, out, u
    torch.cuda.empty_cache()
    return pts / best / 1e6


def write_table(choice, path):
    lines = ["// Generated by `python -m sympygr_amd.autotune` -- do not edit.",
             "// RHS tile shape per interior size: {{nx, ny, nz}, {tx, ty, tz}} (sizes not listed: 8^3)."]
    for n, s in sorted(choice.items()):
        if tuple(s) != (8, 8, 8):
            lines.append(f"{{{{{n}, {n}, {n}}}, {{{s[0]}, {s[1]}, {s[2]}}}}},")
    with open(path, "w") as f:
        f.write("\n".join(lines) + "\n")


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--sizes", type=int, nargs="+", default=[9, 13, 16, 17, 24, 25, 32, 33, 48])
    ap.add_argument("--top", type=int, default=6, help="shapes timed per size besides 8^3")
    ap.add_argument("--dry-run", action="store_true", help="list the candidates only (no GPU)")
    ap.add_argument("--table", default=TABLE, help="where to write the tile table")
    ap.add_argument("--report", default=REPORT, help="where to write the timings")
    args = ap.parse_args()
    if args.dry_run:
        for n in args.sizes:
            print(n, [(s, round(cost(n, s), 2)) for s in candidates(n, args.top)])
        return
    git = subprocess.run(["git", "rev-parse", "--short", "HEAD"], capture_output=True, text=True,
                         cwd=ROOT).stdout.strip() or None  # None outside a git checkout
    report = {"git": git, "metric": "RHS Mpoints/s, mixed precision, upwind, uniform tiling of n^3 blocks (about 12 M points)",
              "sizes": {}}
    choice = {}
    for n in args.sizes:
        res = {}
        for s in candidates(n, args.top):
            r = time_shape(n, s)
            res["x".join(str(x) for x in s)] = r
            print(f"[autotune] n={n} shape={s}: {r:.1f} Mpts/s", flush=True)
        best = max(res, key=res.get)
        choice[n] = tuple(int(x) for x in best.split("x"))
        report["sizes"][str(n)] = {"timings": res, "best": best, "gain_vs_8cubed": res[best] / res["8x8x8"]}
        print(f"[autotune] n={n}: {best} ({res[best] / res['8x8x8']:.2f}x of 8^3)", flush=True)
    write_table(choice, args.table)
    with open(args.report, "w") as f:
        json.dump(report, f, indent=1)
    print(f"wrote {args.table} and {args.report}")


if __name__ == "__main__":
    sys.exit(main())
