"""The buffer descriptors of both kernels' tiles (partition_map.h: tile_base, tile_bytes, tile_row_offset; 16 tokens, FP32
4): for every position of a range's end in a tile, the rows inside the descriptor are the live ones, each lies in its
page, and a tile that is not live has no bytes. A tile of the window names the window entry of its page; one past the
window, which ends the range, is not live."""
import subprocess


from gpu_util import no_child_processes_after_gpu_init
from test_address_audit import CSRC, compiler

SOURCE = r"""
#include <stdio.h>
#include <initializer_list>
#include "partition_map.h"
using namespace pd;
int main() {
    long checks = 0, bad = 0;
    for (int tokens : {kTileTokens, kFp32TileTokens})
    for (int page_shift = 4; page_shift <= 5; ++page_shift)
        for (uint32_t head_bytes : {64u, 128u, 256u, 512u})
            for (int heads : {1, 5, 8}) {
                PartialParams p{};
                p.page_shift = page_shift;
                p.physical_pages = 0x7FFFFFFF;
                p.token_bytes = heads * head_bytes;
                p.page_bytes = (1ull << page_shift) * p.token_bytes;
                for (int page : {0, 1, 70000, 0x7FFFFFFE, -1, 0x7FFFFFFF})
                    for (int t0 = 0; t0 < 96; t0 += tokens)
                        for (int re = 0; re <= t0 + 40; ++re) {
                            const bool ok = tile_live(p, t0, re, page);
                            const uint64_t bytes = tile_bytes(p, ok, t0, re, tokens);
                            for (int row = 0; row < tokens; ++row)
                                for (uint32_t lane = 0; lane < head_bytes; lane += 16, ++checks) {
                                    const bool read = tile_row_offset(p, row, lane) < bytes;  // the hardware's check
                                    const bool live = page >= 0 && page < p.physical_pages && t0 + row < re;
                                    bad += read != live;
                                    const int slot = (t0 + row) % (1 << page_shift);
                                    if (read)
                                        bad += tile_base(p, page, t0) + tile_row_offset(p, row, lane) !=
                                               static_cast<uint64_t>(page) * p.page_bytes + slot * p.token_bytes + lane;
                                }
                        }
            }
    for (int tokens : {kTileTokens, kFp32TileTokens})
        for (int page_shift = 4; page_shift <= 5; ++page_shift)
            for (int window : {0, 1, 7, 200}) {
                PartialParams p{};
                p.page_shift = page_shift;
                p.physical_pages = 0x7FFFFFFF;
                const int end = (window + kWave) << page_shift;  // the range of a window ends with it
                for (int t0 = window << page_shift; t0 < end + 64; t0 += tokens, ++checks) {
                    const int slot = tile_slot(p, t0, window);
                    bad += t0 < end ? slot != (t0 >> page_shift) - window : slot != kWave - 1;
                    bad += tile_live(p, t0, end, 0) != (t0 < end);
                }
            }
    printf("%ld checks, %ld bad\n", checks, bad);
    return bad != 0;
}
"""


def test_tile_descriptors_hold_the_live_rows(tmp_path):
    no_child_processes_after_gpu_init()
    source, exe = tmp_path / "tiles.cpp", tmp_path / "tiles"
    source.write_text(SOURCE)
    subprocess.run([compiler("g++"), "-std=c++17", "-O1", f"-I{CSRC}", str(source), "-o", str(exe)], check=True,
                   capture_output=True, text=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and ", 0 bad" in run.stdout, run.stdout
