"""Batched 2-D ensemble: barriers where waves of a workgroup run different loops,
and the edge of the workgroup."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "masterthesis_amd", "csrc",
                   "batch2d.hip")


def test_no_block_barrier_in_the_loops_that_waves_choose_between():
    """__syncthreads wants every thread at the same call; the masked and the plain
    loop each have their own, so they use the wave-counting barrier instead, in
    equal numbers because both are one body."""
    src = open(SRC).read()
    body = re.search(r"auto steps = \[&\].*?\n    \};\n", src, re.S).group(0)
    assert "__syncthreads" not in body and body.count("wave_barrier()") == 2
    assert re.search(r"if \(plain\) steps\(false\);\s*else steps\(true\);", src)
