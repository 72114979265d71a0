"""Host rules of the LJ kernels' launches, compiled for the host alone and run
without a device."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(tmp_path, body):
    """the output of a host program with the LJ kernels' header and this main(),
    linked with the library"""
    from pairs_amd import build
    src, exe = tmp_path / "main.cpp", tmp_path / "main"
    src.write_text('#include "%s/pairs_amd/csrc/md_kernels.hpp"\n#include <cstdio>\nusing namespace pk;\n'
                   "int main() {\n%s\n}\n" % (ROOT, body))
    subprocess.run([build.hipcc(), "-O1", "-std=c++17", "-x", "hip", "--offload-host-only", "--offload-arch=gfx950",
                    "-Wno-unused-result", str(src), "-o", str(exe), "-L" + build.HERE, "-lpairs_hip",
                    "-Wl,-rpath," + build.HERE], check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout


@pytest.mark.parametrize("nlocal,gmax", [(200000, 4000), (200064, 1563), (200065, 1564), (1048576, 26970)])
def test_tile_table_before_a_build(tmp_path, nlocal, gmax):
    """the force kernel reads every row of the table: all locals once, the rest empty"""
    out = _run(tmp_path, "for (const int4 &t : tiles_before_build(%d, %d)) printf(\"%%d %%d %%d\\n\", t.x, t.y, t.z);"
               % (nlocal, gmax))
    rows = [tuple(map(int, l.split())) for l in out.splitlines()]
    assert len(rows) == gmax
    at = 0
    for first, count, size in rows:
        assert size == 0 and 0 <= count <= 128
        if count:
            assert first == at
            at += count
    assert at == nlocal


def test_idle_lanes_of_a_tile_walk_rows_of_their_wave(tmp_path):
    """a local's 16-bit rows are padded to the depth of the wave that it is in"""
    out = _run(tmp_path, "for (int n = 1; n <= TILE_G; n++) for (int t = 0; t < TILE_G; t++) "
                         "printf(\"%d %d %d\\n\", n, t, tile_lane_row(t, n));")
    for l in out.splitlines():
        n, t, r = map(int, l.split())
        assert 0 <= r < n and (r == t or t >= n)
        # (a wave without a local has no entry to walk)
        assert r // 64 == t // 64 or n <= t // 64 * 64


def test_build_workgroup_fits_the_lds(tmp_path):
    """whatever the length of the columns, the tile and the list form: a build that
    fits a workgroup of two waves is launched in one that fits"""
    out = _run(tmp_path, """
    for (int nz = 4; nz < 1300; nz += 7) for (int half = 0; half < 2; half++) for (int chunks = 1; chunks < 3; chunks++)
    for (int cap : {64, 640, 4096, 8192, 8256, 30000}) for (int n : {300, 79999, 80001}) {
        DevState d{};
        Geom g{};
        d.max_lds = 163840; d.nlocal = n; d.tile_cap = cap;
        g.dim_cells[0] = g.dim_cells[1] = 7; g.dim_cells[2] = nz; g.nchunks = chunks; g.zc = nz / chunks;
        if (build_tile_limit(d, g, half) < 64) continue;
        const int t = build_threads(d, g, half);
        printf("%d %zu %d\\n", t, build_lds_bytes(d, g, half, t), d.max_lds);
    }""")
    rows = [tuple(map(int, l.split())) for l in out.splitlines()]
    assert {t for t, _, _ in rows} == {128, 512}
    for threads, lds, most in rows:
        assert lds + 512 <= most, (threads, lds)  # (less than 512 bytes of static LDS)


def test_tile_places_of_overlapping_runs(tmp_path):
    """cells with many empty ones, columns no longer than a group: a slot of any
    candidate run has a place, and the place is the slot's"""
    out = _run(tmp_path, """
    unsigned seed = 1;
    auto rnd = [&](int n) { seed = seed * 1664525u + 1013904223u; return (int) ((seed >> 8) % (unsigned) n); };
    int equal = 0, wrong = 0, slots = 0;
    for (int c = 0; c < 4000; c++) {
        const int nx = 3 + rnd(3), ny = 3 + rnd(3), nz = 3 + rnd(6), ncells = nx * ny * nz + 1, fill = 1 + rnd(12);
        std::vector<int> at[2];  // first slots of the cells: locals, ghosts
        int n = 0;
        for (int k = 0; k < 2; k++) {
            at[k].resize(ncells + 1);
            for (int i = 0; i < ncells; i++) { at[k][i] = n; n += rnd(12) < fill ? rnd(5) : 0; }
            at[k][ncells] = n;
        }
        const int cx = rnd(nx), cy = rnd(ny), za = rnd(nz), zb = za + 1 + rnd(nz - za);
        int start[NRUNS], off[NRUNS + 1] = {0};
        for (int t = 0; t < NRUNS; t++) {
            int lo = 0, hi = 0;
            if (t >= 2) {
                const int col = (t - 2) / 2, B = ((cx + col / 3 - 1) * ny + cy + col % 3 - 1) * nz + 1;
                lo = std::max(B + za - 1, 1);
                hi = std::min(B + zb, ncells - 1);
            }
            start[t] = lo <= hi ? at[t & 1][lo] : 0;
            off[t + 1] = off[t] + (lo <= hi ? at[t & 1][hi + 1] - start[t] : 0);
        }
        int from[32], delta[32] = {0};
        for (int &f : from) f = 0x7fffffff;
        for (int t = 0; t < NRUNS; t++) {
            if (off[t + 1] == off[t]) continue;
            const int r = tile_run_rank(start, off, t);
            from[r] = start[t];
            delta[r] = off[t] - start[t];
            for (int k = 0; k < t; k++) equal += off[k + 1] > off[k] && start[k] == start[t];
        }
        for (int t = 0; t < NRUNS; t++)
            for (int j = start[t]; j < start[t] + off[t + 1] - off[t]; j++) {
                const int p = tile_place(from, delta, j);
                bool ok = false;
                for (int r = 0; r < NRUNS; r++) ok = ok || (p >= off[r] && p < off[r + 1] && start[r] + p - off[r] == j);
                wrong += !ok;
                slots++;
            }
    }
    printf("%d %d %d\\n", equal, wrong, slots);""")
    equal, wrong, slots = map(int, out.split())
    assert equal > 100 and slots > 10000
    assert wrong == 0, (wrong, slots)
