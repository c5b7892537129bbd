"""bench.py's work per padded cell against a count of the cells that the kernels
visit: a path runs from its border to its last crop cell, the fused sweep from
its first row to its last crop row, the WTA over every row that is not a copy
of a padding band's first one."""
import pytest

import bench


@pytest.mark.parametrize("shapes", [[(12, 8, 8)], [(8, 20, 16)], [(4, 4, 24)], [(12, 8, 8), (20, 12, 16)]])
def test_work_per_cell_counts_visited_cells(shapes):
    total = 0
    n = dict.fromkeys(("rows", "paths", "sweep", "wta", "crop"), 0)
    for W, H, D in shapes:
        Wp, Hp = W + 2 * D, H + 2 * D
        crop = {(x, y) for x in range(D, D + W) for y in range(D, D + H)}
        for dx, dy in ((1, 0), (-1, 0), (0, 1), (0, -1), (1, 1), (-1, -1), (1, -1), (-1, 1)):
            seen = set()
            for x, y in crop:
                while 0 <= x < Wp and 0 <= y < Hp:   # against the path, to its border
                    seen.add((x, y))
                    x, y = x - dx, y - dy
            n["paths"] += len(seen) * D
            n["rows"] += len(seen) * D if dy == 0 else 0
        n["sweep"] += 2 * Wp * len(range(D + H)) * D
        for R, C in ((Hp, Wp), (Wp, Hp)):
            own = [r for r in range(R) if not (3 < r <= D - 4 or R - D + 3 < r <= R - 4)]
            n["wta"] += len(own) * C * D / 2   # two frames of each shape, 28 ops for all four
        n["crop"] += len(crop) * D
        total += Wp * Hp * D
    work, crop = bench.kernel_work([dict(W=W, H=H, D=D) for W, H, D in shapes])
    assert crop == pytest.approx(n["crop"] / total)
    want = {"wta": (28 * n["wta"], None), "msum": (4 * total, total), "sgm_rows": (8 * n["rows"], n["rows"] + n["crop"]),
            "sgm_vsweep": (24 * n["sweep"] + n["crop"], n["sweep"] + 5 * n["crop"]), "sgm_paths": (8 * n["paths"], None),
            "winner": (n["crop"], None)}
    assert set(work) == set(want)
    for k, (ops, byt) in want.items():
        assert work[k][0] == pytest.approx(ops / total), k
        assert work[k][1] is None if byt is None else work[k][1] == pytest.approx(byt / total), k


def test_roofline_prices_the_computed_work():
    """A batch on the fused sweep: the step and its dominant kernel."""
    rigs = [dict(W=1920, H=1080, D=192)] * 2
    cells = 2 * 2304 * 1464 * 192
    work, _ = bench.kernel_work(rigs)
    kern = {"wta": 1.0, "msum": 1.0, "sgm_rows": 1.0, "sgm_vsweep": 4.0}
    r = bench.roofline_entry(kern, {"sgm_vsweep": 160}, cells, 8.0, 2, "mixed", rigs)
    ops = sum(work[k][0] for k in kern)
    assert r["ops_per_cell"] == 97 and r["ops_per_cell_computed"] == pytest.approx(ops)
    assert r["frac_computed"] == pytest.approx(ops * cells / 8e-3 / bench.VALU_PEAK)
    d = r["dominant_kernel"]
    assert d["kernel"] == "sgm_vsweep"
    assert d["frac"] == pytest.approx(work["sgm_vsweep"][0] * cells / 4e-3 / bench.VALU_PEAK)
    assert d["bytes_per_cell"] == pytest.approx(work["sgm_vsweep"][1])
    assert d["hbm_frac"] == pytest.approx(work["sgm_vsweep"][1] * cells / 4e-3 / bench.HBM_PEAK)
