"""The MFMA down's units against the same rows alone (GPU).

A unit of the routed down holds 16 or 32 rows of the list of a pick batch's experts' tile rows
(28, 20 or 4 a tile), so it may hold rows of several experts and meet the picks of all of them;
each value kept is one expert's row against that expert's pick, whose sum no other row, pick or
unit enters. A step's rows must therefore come out as each row does by itself, bit for bit, on the
converting MFMA and on the scaled one (MXFP4; by default from 8 rows where inter <= 512): one
row has 6 or 8 experts with one pick each (one unit boundary in each second expert at most), a
step of many rows every cut of a tile, several pick batches, experts split over two of them and,
with skewed routing, experts with more picks than an MFMA's 16 columns.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu


CASES = [
    ("plumbing_fp8", "row_major", 17, 0.0),  # 4-row tiles: up to five experts a unit
    ("dsv3_tp4_fp8", "row_major", 2, 0.0),
    ("dsv3_tp4_fp8", "row_major", 16, 0.0),  # 128 picks: two batches of 64
    ("dsv3_tp4_fp8", "row_major", 48, 1.2),
    ("dsv3_tp4_mxfp4", "row_major", 9, 0.0),
    ("dsv3_tp4_mxfp4", "aiter", 3, 0.0),
    ("dsv3_tp4_mxfp4", "aiter", 48, 1.2),
    ("dsv3_tp2_mxfp4_norm", "row_major", 8, 0.0),  # 64 picks: two batches of 32
    ("dsv3_tp2_mxfp4_norm", "aiter", 16, 1.2),
    ("v41_tp4", "aiter", 2, 0.0),
    ("v41_tp4", "aiter", 13, 0.0),  # 78 picks: two batches of 39
    ("v41_tp4", "aiter", 25, 0.0),  # 150 picks: two whole batches of 75, the second's scales off a piece's start
    ("v41_tp4", "aiter", 48, 1.2),
    ("v41_tp2", "aiter", 9, 0.0),  # 54 picks: two batches of 27
    ("v41_tp2", "aiter", 33, 1.2),
]


# MXFP4: the converting MFMA and the scaled one; FP8 has one
@pytest.mark.parametrize(
    "preset,layout,rows,zipf,scaled", [(*c, s) for c in CASES for s in (False, True) if not (s and "fp8" in c[0])]
)
def test_rows_do_not_depend_on_the_step(preset, layout, rows, zipf, scaled):
    from bench import make_layer
    from sgl_amd_mono.moe.presets import PRESETS
    from sgl_amd_mono.moe.runner import MoeRunner

    p = PRESETS[preset]
    g = torch.Generator(device="cuda").manual_seed(97 + rows)
    w = make_layer(p, g, "cuda", zipf)
    x = torch.randn(rows, p.hidden, generator=g, device="cuda").to(torch.bfloat16)
    x[:, 0] = 1.0
    # (one MFMA at every row count, where the default chooses by it)
    run = MoeRunner(p, layout=layout, mxfp4_scaled_down_rows=1 if scaled else 49)
    out = run.moe(w, x)
    for r in range(rows):
        alone = run.moe(w, x[r : r + 1])
        assert torch.equal(out[r], alone[0]), f"row {r} of {rows}"
    run.raise_on_device_error()
    for polled in ("router_parts_polled", "picks_polled"):  # left unset for the next launch
        assert bool((run.region(polled) == 0xFF).all()), polled
    assert torch.isfinite(out.float()).all() and out.float().abs().max() > 0
