"""The order of memory operations in gemm_block's K loop, on the CPU: the
kernel issues its LDS reads and DMAs from gemm_block_order.h, and a host program
walks the same functions. Four waves meet at one barrier per unit; a wave's
reads return in order and its DMAs complete in order, at any time before the
wait that covers them. So

- a DMA may land at once: every read, by any wave, of the LDS it overwrites has
  to have returned before the barrier at the top of the unit that issues it;
- a DMA may land as late as its wait: what a unit reads has to have been waited
  for, by the wave that issued it, before the barrier at the top of that unit.
"""
import pathlib
import subprocess

import pytest

KERNELS = pathlib.Path(__file__).resolve().parent.parent / "cu-jev_amd" / "csrc" / "kernels"

WALK = r"""
#include "gemm_block_order.h"
#include <cstdio>
#include <vector>

struct Op { int unit, buf, data; }; /* unit that issues it, LDS region, what is in it */

static int bad;
static void fault(const char *what, int WN, int unit, int buf) {
    if (bad++ < 5)
        printf("WN %d unit %d region %d: %s\n", WN, unit, buf, what);
}

/* regions: W ring slots 0..3, X buffers 4 and 5. Every wave issues the same
 * order, and reads what other waves load, so one wave's queues stand for all. */
static void walk(int WN, int units) {
    std::vector<Op> reads, dmas;
    std::vector<size_t> reads_done(units), dmas_done(units), reads_at(units), dmas_at(units);
    auto w = [&](int unit, int u) { dmas.push_back({unit, u & 3, u}); };
    auto x = [&](int unit, int p) { for (int j = 0; j < WN; j++) dmas.push_back({unit, 4 + (p & 1), p}); };
    /* prologue, as unit -1 */
    x(-1, 0);
    for (int u = 0; u < 2; u++) for (int k = 0; k < 4; k++) w(-1, u);
    x(-1, 1);
    for (int k = 0; k < 4; k++) w(-1, 2);
    const size_t first = dmas.size() - (WN + 4); /* what its wait covers */
    for (int j = 0; j < WN; j++) reads.push_back({-1, 4, 0});
    for (int r = 0; r < GB_AD; r++) reads.push_back({-1, 0, 0});
    for (size_t i = first; i < dmas.size(); i++)
        for (auto &rd : reads)
            if (dmas[i].buf == rd.buf && dmas[i].data == rd.data)
                fault("prologue reads before its wait", WN, -1, rd.buf);
    for (int u = 0; u < units; u++) {
        const int S = u & 3;
        reads_at[u] = reads.size(), dmas_at[u] = dmas.size();
        const size_t lg = gb_lgkm(S, WN), vm = gb_vm(S, WN);
        reads_done[u] = reads.size() > lg ? reads.size() - lg : 0;
        dmas_done[u] = dmas.size() > vm ? dmas.size() - vm : 0;
        int na = 0, nb = 0, nw = 0, nx = 0;
        for (int r = 0; r < 8; r++)
            for (int j = 0; j < WN; j++) {
                const gb_mem m = gb_before(S, WN, r, j);
                const int un = m.slot == S ? u : u + 1; /* the unit a read is for */
                if (m.kind == GB_READ_A) {
                    if (m.row != ((r + GB_AD) & 7) || (un & 3) != m.slot) fault("W row", WN, u, m.slot);
                    reads.push_back({u, m.slot, un}), na++;
                }
                if (m.kind == GB_READ_B) {
                    if (m.row != nb || m.slot != ((u + 1) & 3)) fault("X row", WN, u, m.slot);
                    reads.push_back({u, 4 + (m.slot >> 1), (u + 1) >> 1}), nb++;
                }
                if (m.kind == GB_DMA_W) {
                    if (m.row != nw || m.slot != ((u + 3) & 3)) fault("W piece", WN, u, m.slot);
                    w(u, u + 3), nw++;
                }
                if (m.kind == GB_DMA_X) {
                    if (m.row != nx || m.slot >> 1 != (((u >> 1) + 2) & 1)) fault("X piece", WN, u, m.slot);
                    dmas.push_back({u, 4 + (m.slot >> 1), (u >> 1) + 2}), nx++;
                }
            }
        if (na != 8 || nb != WN || nw != 4 || nx != (S & 1 ? WN : 0)) fault("count", WN, u, 0);
        /* reads of this unit: the data is there, and nothing later was sent to its place */
        for (size_t i = reads_at[u]; i < reads.size(); i++) {
            bool there = false;
            for (size_t d = 0; d < dmas.size(); d++) {
                if (dmas[d].buf != reads[i].buf) continue;
                if (dmas[d].data == reads[i].data) {
                    there = true;
                    if (d >= dmas_done[u]) fault("read of a piece not waited for", WN, u, reads[i].buf);
                } else if (dmas[d].data > reads[i].data) {
                    fault("read of a place that is being overwritten", WN, u, reads[i].buf);
                }
            }
            if (!there) fault("read of what was never loaded", WN, u, reads[i].buf);
        }
        /* DMAs of this unit: no earlier read of the place may be outstanding */
        for (size_t d = dmas_at[u]; d < dmas.size(); d++)
            for (size_t i = reads_done[u]; i < reads_at[u]; i++)
                if (reads[i].buf == dmas[d].buf) fault("overwrites a read in flight", WN, u, dmas[d].buf);
    }
}

int main() {
    for (int WN = 4; WN <= 8; WN += 2) walk(WN, 24);
    return bad ? 1 : 0;
}
"""


@pytest.mark.parametrize("wait", ["as built", "one read too many", "one DMA too many"])
def test_units_are_ordered_by_their_waits(tmp_path, wait):
    """The planted waits show that the walk sees what it is there for."""
    order = (KERNELS / "gemm_block_order.h").read_text()
    if wait == "one read too many":
        assert "? 3 : 4" in order
        order = order.replace("? 3 : 4", "? 4 : 4")
    if wait == "one DMA too many":
        assert "? 4 : 4 + WN" in order
        order = order.replace("? 4 : 4 + WN", "? 5 : 4 + WN")
    (tmp_path / "gemm_block_order.h").write_text(order)
    (tmp_path / "walk.cpp").write_text(WALK)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-o", "walk", "walk.cpp"], cwd=tmp_path,
                   check=True)
    r = subprocess.run(["./walk"], cwd=tmp_path, capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == (0 if wait == "as built" else 1), r.stdout
