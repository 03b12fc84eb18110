"""Measures, on an MI355X, how torch.nn.functional.linear (hipBLASLt) splits the
K range of the last output tiles of a bf16 [M, K] x [N, K]^T product, and
writes the table the HIP GEMM uses to accumulate those tiles the same way
(``csrc/streamk_tail.h``).

For some shapes the library runs its last output tiles as a "stream-K" tail:
a 256 x 256 tile's K range is cut at a tile-dependent point s and the two
partial sums (K < s and K >= s) are accumulated separately and then added.
The split is data-independent, so it is read off one product whose inputs
make it visible (``probe_splits``): A is all ones; weight row n holds +2^20 at
the first 32-wide K block, -2^20 at the last, and 2^-4 at one block b(n) in
between.  Summed in one pass the 2^-4 is rounded away next to 2^20 (half an
fp32 ulp, ties to even); it survives only when block b(n) lies in the partial
that begins at s and ends with the -2^20, so per tile the smallest surviving
block is s.  Which tiles split, and where, were checked bitwise against the
library on random inputs (tests/test_gpu_kernels.py).

Usage (needs the GPU):  python -m tiktoktechjam2026track3_amd.streamk_probe 3200000 100000
prints the header to stdout, stamped with the device's CU count and the torch
and HIP versions.  The probe is a maintainer tool: nothing at run time imports
it.  At run time the plugin measures the order of every product shape it runs
the same way (linear_order.py) and registers it with the library; the header's
tables serve C callers that register nothing, on a device like the one they
were measured on.
"""

from __future__ import annotations

import sys
from typing import Dict, Tuple

BLOCK = 32         # K granularity of the probe
TILE = 256         # output tile edge of the library's tail kernel
TAIL_ROWS = 24576  # rows examined at the end of M


def probe_splits(M: int, N: int, K: int, device) -> Dict[Tuple[int, int], int]:
    """{(tile_row, tile_col): s} for every tile whose K range the library
    splits, with s the first K index of the second partial sum."""
    import torch
    import torch.nn.functional as F

    nb = K // BLOCK
    blocks = [1 + (n % (nb - 2)) for n in range(N)]
    w = torch.zeros(N, K, dtype=torch.float32)
    w[:, 0] = 2.0 ** 20
    w[:, K - BLOCK] = -(2.0 ** 20)
    for n in range(N):
        w[n, BLOCK * blocks[n]] = 2.0 ** -4
    w = w.to(device).bfloat16()
    a = torch.ones(M, K, device=device, dtype=torch.bfloat16)
    bias = torch.zeros(N, device=device, dtype=torch.bfloat16)
    out = F.linear(a, w, bias)
    first = max(0, M - TAIL_ROWS)
    kept = (out[first:] != 0).cpu()
    del out, a
    splits: Dict[Tuple[int, int], int] = {}
    for r0 in range((first + TILE - 1) // TILE * TILE, M, TILE):
        rows = kept[r0 - first: min(M, r0 + TILE) - first]
        if not bool((rows == rows[0:1]).all()):
            raise RuntimeError(f"rows of tile row {r0 // TILE} split differently")
        row = rows[0]
        for tc in range(N // TILE):
            survived = sorted({blocks[n] for n in range(tc * TILE, (tc + 1) * TILE) if bool(row[n])})
            if not survived:
                continue
            if survived != list(range(survived[0], nb - 1)):
                raise RuntimeError(f"tile ({r0 // TILE}, {tc}): surviving blocks are not one range: {survived}")
            splits[(r0 // TILE, tc)] = survived[0] * BLOCK
    return splits


def emit_header(tables: Dict[Tuple[int, int, int], Dict[Tuple[int, int], int]], cus: int,
                torch_version: str, hip_version: str) -> str:
    lines = [
        f"// Generated by tiktoktechjam2026track3_amd/streamk_probe.py on an MI355X ({cus} CUs)",
        f"// with torch {torch_version} (HIP {hip_version}) and the hipBLASLt it bundles: the K",
        "// split torch.nn.functional.linear applies to the last 256 x 256 output tiles of",
        "// these bf16 [M, K] x [N, K]^T products.  split[(tile_row - first_tile_row) *",
        "// tile_cols + tile_col] is the first K index of the second partial sum, 0 when",
        "// the tile is accumulated in one pass.  The library applies these tables only on",
        "// a device with kStreamKTablesCUs CUs, and only to shapes for which the host",
        "// registered no measured order (enc_linear_order_register), which the Python",
        "// plugin does for every product it runs.",
        "#pragma once",
        "#include <stdint.h>",
        "",
        "namespace enc {",
        "",
        f"constexpr int kStreamKTablesCUs = {cus};",
        "",
        "struct StreamKTail {",
        "  int64_t m;",
        "  int n, k;",
        "  int first_tile_row, tile_rows, tile_cols;",
        "  const uint16_t* split;",
        "};",
        "",
    ]
    entries = []
    for (M, N, K), splits in sorted(tables.items()):
        first = min(tr for tr, _ in splits)
        last = (M + TILE - 1) // TILE - 1
        cols = N // TILE
        values = [splits.get((tr, tc), 0) for tr in range(first, last + 1) for tc in range(cols)]
        name = f"kTailSplit_{M}_{N}_{K}"
        lines.append(f"constexpr uint16_t {name}[{len(values)}] = {{")
        for i in range(0, len(values), 16):
            lines.append("    " + ", ".join(str(v) for v in values[i:i + 16]) + ",")
        lines.append("};")
        entries.append(f"    {{{M}, {N}, {K}, {first}, {last - first + 1}, {cols}, {name}}},")
    lines += ["", "constexpr StreamKTail kStreamKTails[] = {"] + entries + ["};", "", "}  // namespace enc"]
    return "\n".join(lines) + "\n"


def main(argv=None) -> int:
    import torch

    args = [int(a) for a in (argv if argv is not None else sys.argv[1:])] or [3200000]
    device = torch.device("cuda:0")
    tables = {}
    for M in args:
        tables[(M, 1024, 1024)] = probe_splits(M, 1024, 1024, device)
        torch.cuda.empty_cache()
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    sys.stdout.write(emit_header(tables, cus, torch.__version__, str(torch.version.hip)))
    return 0


if __name__ == "__main__":
    sys.exit(main())
