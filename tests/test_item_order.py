"""The order in which a gather's items are dealt out, on the CPU: the maps of gather_common.h compiled for the host."""
import os
import subprocess
import tempfile

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# argv: triples of column tiles, token tiles, forced column split.  Every item once, a block of token tiles through all of an XCD's
# columns before the next, and positions past the last item -- a workgroup decodes one when it has fetched its last slice -- give a value.
SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include "gather_common.h"
using namespace pimdl;
int main(int argc, char** argv)
{
    for (int a = 1; a + 2 < argc; a += 3) {
        const uint32_t cols = atoi(argv[a]), toks = atoi(argv[a + 1]), forced = (uint32_t)strtoul(argv[a + 2], 0, 10), items = cols * toks;
        const uint32_t grid = items < 512 ? items : 512;
        for (uint32_t tok_block : {1u, 2u, 4u, 8u, 16u}) {
            const XcdMap map = choose_xcd_map(cols, toks, grid, 1u << 20, 1u << 20, forced);
            const XcdBlocks order = xcd_blocks(map, cols, toks, tok_block);
            std::set<uint64_t> seen;
            for (uint32_t lane = 0; lane < (map.col_split ? 8u : 1u); ++lane) {  // an XCD's positions, in order
                const uint32_t stride = map.col_split ? 8 : 1, width = map.col_split ? tok_block : 8 * tok_block;
                uint32_t block = 0, split = map.col_split ? map.tok_split : 1;
                for (uint32_t p = lane; p < items; p += stride) {
                    uint32_t c = ~0u, t = ~0u;
                    order.decode(p, toks, c, t);
                    if (c >= cols || t >= toks || !seen.insert((uint64_t)c << 32 | t).second) return printf("%u x %u, position %u: %u %u\n", cols, toks, p, c, t), 1;
                    const uint32_t b = t / split / width;
                    if (b < block) return printf("%u x %u, position %u: block %u after %u\n", cols, toks, p, b, block), 1;
                    block = b;
                }
            }
            if (seen.size() != items) return printf("%u x %u: %zu items\n", cols, toks, seen.size()), 1;
            for (uint32_t p = items; p < items + 2 * grid; ++p) {
                volatile uint32_t position = p, use;
                uint32_t c, t;
                order.decode(position, toks, c, t);
                use = c + t;
                (void)use;
            }
        }
    }
    printf("ok\n");
}
"""


def test_blocks_of_token_tiles_deal_every_item_once():
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc here")
    plain = 0xFFFFFFFF
    cases = [(64, 128, 0), (43, 64, 0), (42, 69, 0), (32, 94, 0), (32, 94, 8), (24, 128, 4), (16, 256, 2), (8, 16, 1), (1, 513, 0), (1, 1, 0), (3, 7, plain),
             (64, 64, plain), (42, 72, 1), (171, 33, 0), (48, 1000, 0), (7, 4097, 0), (2731, 8, 0)]
    with tempfile.TemporaryDirectory() as d:
        open(os.path.join(d, "t.hip"), "w").write(SOURCE)
        subprocess.check_call([HIPCC, "--offload-host-only", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "include"), "-I",
                               os.path.join(ROOT, "pim-dl-asplos_amd", "csrc"), "-o", os.path.join(d, "t"), os.path.join(d, "t.hip")])
        run = subprocess.run([os.path.join(d, "t")] + [str(v) for c in cases for v in c], capture_output=True, text=True)
    assert run.returncode == 0 and run.stdout.strip() == "ok", (run.returncode, run.stdout, run.stderr)
