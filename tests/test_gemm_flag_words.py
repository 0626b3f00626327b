"""The words in LDS through which one wavefront tells the others which flags it saw: every wavefront has read them before the next wait
writes them, or a late one takes that wait's words for its own, skips the wait and is a barrier out of step.  The gap is
two trips to memory wide, so that no launch shows it; the source does."""

import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "syncopate_amd" / "csrc"


def test_words_are_written_behind_a_barrier():
    source = re.sub(r"//[^\n]*", "", (CSRC / "gemm.hip").read_text())
    begin = source.index("gemm_wave_kernel(const GemmParams p) {")
    kernel = source[begin:source.index("\n}\n", begin)]
    wait = kernel.index("auto wait_flag = [&]() -> bool {")
    first_reads, in_wait = kernel[:wait], kernel[wait:kernel.index("};", wait)]
    word = re.compile(r"\bs_spun\b|\bs_waves_up\b")
    # what is read in front of the walk are other words, or they are read in front of a barrier
    uses = [m.end() for m in word.finditer(re.sub(r"__shared__[^;]*;", lambda m: " " * len(m.group()), first_reads))]
    assert not uses or "__syncthreads()" in first_reads[uses[-1]:]
    # written in front of a wait's first barrier only, read between that and the second
    head, middle, tail = in_wait.split("__syncthreads();")
    assert re.search(r"s_waves_up = ", head) and not re.search(r"s_(spun|waves_up) = ", middle)
    assert word.search(middle) and not word.search(tail)
