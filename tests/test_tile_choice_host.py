"""The 3+1D tile of the mixed form where none was set (vh::mixed_tile_3d): for
every width, a tile whose padded rows are not more than its cells' cost
allows, so that narrow lattices do not run on 16-cell rows that stay empty."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
TX, COST = (16, 6, 8), (1.0, 1.45, 1.21)


def test_narrow_rows_get_narrow_tiles(tmp_path):
    exe = str(tmp_path / "tile_choice_check")
    subprocess.run(["/opt/rocm/bin/hipcc", "--offload-host-only", "-O1", "-std=c++17", "-o", exe,
                    os.path.join(HERE, "tile_choice_check.cpp")], check=True, capture_output=True)
    lines = subprocess.run([exe], capture_output=True, text=True, timeout=60, check=True).stdout.split("\n")
    picks = {tuple(map(int, x.split()[:3])): int(x.split()[3]) for x in lines if x and not x.startswith("mix")}
    assert len(picks) == 140 * 6 * 3
    for (nx, ny, nz), v in picks.items():
        padded = [c * (-(-nx // t) * t) for t, c in zip(TX, COST)]
        assert 0 <= v < 3
        if ny > 5:
            assert padded[v] == min(padded), (nx, ny, nz, v)
        assert picks[nx, ny, 2] == v
    assert all(picks[nx, 65, 33] == 1 for nx in (3, 5, 6, 17, 18))
    assert all(picks[nx, 65, 33] == 2 for nx in (7, 8, 19, 20, 24))
    assert all(picks[nx, 65, 33] == 0 for nx in (16, 31, 32, 48, 101, 128))
    assert picks[101, 5, 33] == 1
    assert [x for x in lines if x.startswith("mix")] == ["mix 0", "mix 1"]
