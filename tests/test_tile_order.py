"""The order of the cells in the tile list (tpm_tile_order.hpp), host code: a bijection with its inverse, and the slots
that find the chunks of crowded cells: together with the waves of a cell's first chunks they make every chunk once."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "tpm_tile_order.hpp"
static int order(int C) {
    const int n = C * C * C;
    std::vector<char> seen(n, 0);
    for (int c = 0; c < n; c++) {
        const int r = tile_rank((unsigned)c, (unsigned)C);
        if (r < 0 || r >= n || seen[r]) return 1;
        seen[r] = 1;
        if (tile_cell((unsigned)r, (unsigned)C) != c) return 2;
    }
    return 0;
}
// chunks of ct tiles of cells with the counts given, slots every `space` tiles, the first `run` chunks by the cells
static int slots(const std::vector<int>& cnt, int space, int ct, int run, int total_slots) {
    std::vector<int> off(cnt.size() + 1, 0);
    std::vector<std::vector<int>> made(cnt.size());
    for (size_t r = 0; r < cnt.size(); r++) {
        off[r + 1] = off[r] + cnt[r];
        made[r].assign((cnt[r] + ct - 1) / ct, 0);
        for (int k = 0; k < run && k * ct < cnt[r]; k++) made[r][k]++;
    }
    for (int v = 0; v < total_slots; v++) {
        if (v * space >= off.back()) break;
        size_t r = 0;
        while (off[r + 1] <= v * space) r++;
        const int k = tile_slot_chunk(v, space, ct, off[r], off[r + 1]);
        if (k >= run) made[r].at(k)++;
    }
    for (auto& m : made)
        for (int k : m)
            if (k != 1) return 1;
    return 0;
}
int main(int argc, char** argv) {
    if (argc == 2) return order(std::atoi(argv[1]));
    const int space = std::atoi(argv[1]), ct = std::atoi(argv[2]), run = std::atoi(argv[3]);
    std::srand(std::atoi(argv[4]));
    for (int trial = 0; trial < 300; trial++) {
        std::vector<int> cnt;
        int total = 0;
        const int cells = 1 + std::rand() % 60;
        for (int i = 0; i < cells; i++) {
            const int kind = std::rand() % 5;
            cnt.push_back(kind == 0 ? 0 : kind == 1 ? 1 : kind == 2 ? std::rand() % (2 * ct) : kind == 3 ? ct * (std::rand() % 9) : std::rand() % 700);
            total += cnt.back();
        }
        if (slots(cnt, space, ct, run, total / space + 1)) return 1;
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "o.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I" + os.path.join(ROOT, "tigerpm_amd", "csrc"), str(d / "o.cpp"),
                    "-o", str(d / "o")], check=True)
    return str(d / "o")


@pytest.mark.parametrize("C", [3, 4, 5, 7, 8, 9, 11, 15, 16, 17, 22, 45, 91, 182])
def test_order_and_inverse(driver, C):
    assert subprocess.run([driver, str(C)]).returncode == 0


@pytest.mark.parametrize("space,ct", [(2, 2), (2, 4), (4, 8), (8, 8), (8, 16), (16, 16), (16, 32)])
@pytest.mark.parametrize("run", [1, 4, 12])
def test_slots_make_every_chunk_once(driver, space, ct, run):
    assert subprocess.run([driver, str(space), str(ct), str(run), "7"]).returncode == 0
