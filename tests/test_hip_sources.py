"""What the kernels' sources have to say themselves, as the compiler does not look into
assembly that is written in them."""

import re
from pathlib import Path

import pytest

HIP = Path(__file__).resolve().parent.parent / "mlx_sharding_amd" / "ops" / "hip"
SOURCES = sorted(p for p in (*HIP.glob("*.hip"), *HIP.glob("*.h")) if not p.stem.endswith("_hip"))


def instructions(source):
    """Of each piece of assembly, its instructions one after the other."""
    for piece in re.findall(r"\basm\b(?:\s+volatile)?\s*\(\s*((?:\"(?:[^\"\\]|\\.)*\"\s*)+)", source):
        text = "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", piece))
        yield [i.strip() for i in re.split(r"\\n|;", text.replace("\\t", " ")) if i.strip()]


@pytest.mark.parametrize("path", SOURCES, ids=lambda p: p.name)
def test_a_load_to_lds_waits_for_its_place(path):
    """A write of M0 by the scalar unit, one instruction at least, then the load to LDS."""
    for piece in instructions(path.read_text()):
        for i, one in enumerate(piece):
            if "_lds_" in one or one.endswith(" lds"):
                # where the place is written elsewhere, nobody knows how far before
                wrote = [k for k in range(i) if re.match(r"s_\w+ m0\b", piece[k])]
                assert wrote and i - wrote[-1] >= 2, (path.name, piece)


@pytest.mark.parametrize("path", SOURCES, ids=lambda p: p.name)
def test_a_barrier_says_what_lies_before_it(path):
    """Behind a barrier in assembly others load into places that this wave has read: its reads
    have returned, in the same piece, or by a wait or a fence that the compiler keeps beside it."""
    text = path.read_text()
    for at in re.finditer(r"asm volatile\(\s*\"[^\"]*s_barrier", text):
        before = text[:at.start()].splitlines()[-2:]
        assert ("s_waitcnt" in at.group() or any("amdgcn_s_waitcnt" in line
                                                 or "amdgcn_sched_barrier" in line
                                                 for line in before)), path.name
