"""CPU checks of the SSD backward's host logic: the chunk table over the scan's
sequences (one row per 64-token chunk, rows of a sequence consecutive, each row
(sequence, first token, end token, 0, 1, index, first row, rows)), the sequence
layout shared by the forward and the backward, and the library's launch rules
(csrc/ssd_backward_plan.hpp, compiled here for the host)."""
import ctypes
import subprocess
from pathlib import Path

import pytest
import torch

from hmx.ops.ssd import seq_layout
from hmx.ops.ssd_train import _chunk_table


def test_chunk_table_tiles_every_sequence():
    bounds = [(0, 130), (130, 130), (130, 131), (300, 428)]
    rows, seqs = _chunk_table(bounds)
    assert rows == [(0, 0, 64, 0, 1, 0, 0, 3), (0, 64, 128, 0, 1, 1, 0, 3),
                    (0, 128, 130, 0, 1, 2, 0, 3),
                    (2, 130, 131, 0, 1, 0, 3, 1),
                    (3, 300, 364, 0, 1, 0, 4, 2), (3, 364, 428, 0, 1, 1, 4, 2)]
    assert seqs == [(0, 3), (3, 0), (3, 1), (4, 2)]
    # every token of every sequence in exactly one row
    covered = sorted(t for r in rows for t in range(r[1], r[2]))
    assert covered == [t for a, e in bounds for t in range(a, e)]


def test_seq_layout_rows_and_restarts():
    seq_idx = torch.tensor([[0, 0, 1, 1, 1], [4, 4, 4, 4, 4]])
    bounds, first, last, end_at = seq_layout(2, 5, seq_idx)
    assert bounds == [(0, 2), (2, 5), (5, 10)]
    assert first == [0, 2] and last == [1, 2]
    assert end_at == {(0, 2): 0, (0, 5): 1, (1, 5): 2}
    bounds, first, last, _ = seq_layout(3, 4)
    assert bounds == [(0, 4), (4, 8), (8, 12)] and first == [0, 1, 2] and last == [0, 1, 2]


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    csrc = Path(__file__).resolve().parent.parent / "hybrid-model-factory_amd" / "csrc"
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text('''
#include "ssd_backward_plan.hpp"
using namespace hmx::ssdb;
extern "C" void blocks(int nrows, int units, int cus, int* out) {
  const StateBlocks b = state_blocks(nrows, units, cus);
  out[0] = b.rows;
  out[1] = b.blocks;
}
extern "C" int group(int G, int GC, int z, const int64_t* ts, int64_t dx_ts, uint64_t dx) {
  return takes_group_kernel(G, GC, z != 0, ts[0], ts[1], ts[2], ts[3], dx_ts, dx);
}
''')
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{csrc}", "-o",
                    str(d / "rules.so"), str(d / "rules.cpp")], check=True)
    return ctypes.CDLL(str(d / "rules.so"))


@pytest.mark.parametrize("cus", [32, 64, 256, 304])
def test_state_blocks_fill_the_device(rules, cus):
    """The table rows are cut just far enough for a workgroup per CU, into blocks that tile
    them, of which the workspace holds at most rows / 8."""
    out = (ctypes.c_int * 2)()
    for nrows in [0, 1, 7, 8, 15, 16, 17, 63, 64, 100, 512, 513, 4096]:
        for units in [2, 4, 24, 62, 64, 66, 128, 254, 256, 258, 512]:
            rules.blocks(nrows, units, cus, out)
            rows, blocks = out
            assert rows >= 1 and blocks >= 1 and rows * blocks >= nrows
            assert blocks == 1 or (rows * (blocks - 1) < nrows and 8 * blocks <= nrows)
            if units >= cus:
                assert blocks == 1, "the heads alone fill the device: no cut"
            elif nrows >= 4096:
                assert units * blocks >= cus * 0.9


def test_group_kernel_takes_what_it_can_address(rules):
    def group(G=4, GC=4, z=0, ts=(512, 512, 512, 512), dx_ts=512, dx=1 << 20):
        return rules.group(G, GC, z, (ctypes.c_int64 * 4)(*ts), ctypes.c_int64(dx_ts),
                           ctypes.c_uint64(dx))

    assert group() and group(ts=(0, 0, 0, 0)) and group(G=1, GC=1)
    assert not group(G=2) and not group(z=1)
    far = (1 << 24) - 8
    for i in range(4):      # a chunk's last row stays within 31-bit byte offsets
        at = lambda v: group(ts=tuple(v if j == i else 512 for j in range(4)))
        assert at(far) and 63 * far * 2 + 2 * 128 <= 1 << 31
        assert not at(far + 8) and not at(1 << 26) and not at(1 << 32) and not at(-8)
    assert group(dx_ts=(1 << 23) - 128) and not group(dx_ts=1 << 23)
    for off in (2, 4, 8):   # dx leaves in pieces of up to 16 bytes
        assert not group(dx=(1 << 20) + off)
    assert group(dx=(1 << 20) + 16)
