"""Writes the GEMM tile-choice table (csrc/kea_gemm_table.h) and its summary (profiles/gemm_tile_sweep.md) from the
output of `python bench.py --sweep 1,2,3` (one JSON line per (wbits, parts, M, N, K) with every tile's per-launch
microseconds on MI355X).

    python kea-kernels_amd/csrc/gen_tile_table.py SWEEP_LOG [SWEEP_LOG ...]

Several logs (for instance one per weight width, `--sweep-wbits 1` and `--sweep-wbits 2`) are merged; a shape swept in
more than one keeps its line from the last log that holds it.

The table keeps, for every swept shape, the fastest tile; the library picks the entry of the same weight width,
part count, N and K with the nearest M in log scale (as the reference's configs.choose does over its tuned points,
kk/binary/configs.py:53-58), and for shapes it does not list, the nearest entry in (log M, log N, log K).
"""
from __future__ import annotations

import json
import sys
from collections import defaultdict
from pathlib import Path

HERE = Path(__file__).resolve().parent
ROOT = HERE.parents[1]


def main(log_paths: list[str]) -> None:
    by_shape = {}
    for log_path in log_paths:
        for line in Path(log_path).read_text().splitlines():
            if line.startswith("{"):
                r = json.loads(line)
                by_shape[(r["wbits"], r["parts"], r["M"], r["N"], r["K"])] = r
    rows = list(by_shape.values())
    entries = []
    groups = defaultdict(list)
    for r in rows:
        times = {int(k[1:]): v for k, v in r.items() if k.startswith("t") and k[1:].isdigit()}
        best = min(times, key=times.get)
        entries.append((r["wbits"], r["parts"], r["N"], r["K"], r["M"], best))
        groups[(r["wbits"], r["parts"], r["N"], r["K"])].append((r["M"], best, times[best], times.get(r["chosen"])))
    entries.sort()
    lines = [f"    {{{w}, {p}, {n}, {k}, {m}, {t}}}," for w, p, n, k, m, t in entries]
    (HERE / "kea_gemm_table.h").write_text(
        "// GEMM tile choice measured on MI355X: the fastest tile id (1-based ids of kea_config_name) for each swept\n"
        "// (weight bits, parts, N, K, M), fp16 scales and output, HIP-graph replay. Generated by gen_tile_table.py\n"
        "// from `bench.py --sweep 1,2,3`; do not edit by hand.\n"
        "#pragma once\n\nnamespace kea {\n\nstruct TileChoice {\n    int wbits, parts, n, k, m, tile;\n};\n\n"
        "constexpr TileChoice kTileTable[] = {\n" + "\n".join(lines) + "\n};\n"
        "constexpr int kTileTableSize = sizeof(kTileTable) / sizeof(kTileTable[0]);\n\n}  // namespace kea\n")
    out = ["# GEMM tile sweep (the chooser table's source)", "",
           "Command (from the repository root on the MI355X box):", "",
           "    python3 bench.py --sweep 1,2,3 --sweep-wbits 1 > sweep1.log",
           "    python3 bench.py --sweep 1,2,3 --sweep-wbits 2 > sweep2.log",
           "    python3 kea-kernels_amd/csrc/gen_tile_table.py sweep1.log sweep2.log", "",
           "Every tile configuration of the library at each (weight bits, parts, N, K, M), fp16 scales and output, "
           "HIP-graph replay of 100 launches (10 above M = 1000) behind a spin, per-launch microseconds. Per row: for each swept M, the "
           "fastest tile `t<id>` and its time; in brackets the time of the tile that the chooser of the swept build "
           "picked, where that was more than 5% slower. Tile ids: 1-12 and 24 on the LDS-ring tiles, "
           "13-23 the wave-split tiles (`kea_config_name`).", "",
           "| bits | P | N | K | M: best tile, us [swept build's choice] |", "|---|---|---|---|---|"]
    for (w, p, n, k), items in sorted(groups.items()):
        cells = []
        for m, best, t, prev in sorted(items):
            c = f"{m}: t{best} {t:.2f}"
            if prev is not None and prev > 1.05 * t:
                c += f" [{prev:.2f}]"
            cells.append(c)
        out.append(f"| {w} | {p} | {n} | {k} | " + "; ".join(cells) + " |")
    tot_best = sum(t for items in groups.values() for _, _, t, _ in items)
    tot_prev = sum(pv for items in groups.values() for _, _, _, pv in items if pv is not None)
    out += ["", f"Sum over the {len(rows)} shapes: {tot_best:.1f} us with the table's tiles, {tot_prev:.1f} us with "
                f"the swept build's choices."]
    (ROOT / "profiles" / "gemm_tile_sweep.md").write_text("\n".join(out) + "\n")
    print(f"{len(entries)} entries; best {tot_best:.1f} us, previous {tot_prev:.1f} us")


if __name__ == "__main__":
    main(sys.argv[1:])
