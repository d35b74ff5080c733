"""Rules of the HIP sources that neither the compiler nor a run would report.

A vector instruction that reads an MFMA's result has to follow it at a
distance; the hardware does not check it, and the compiler puts the wait
states only before instructions of its own.  So inline assembly holds no
vector instructions: barriers, waits and empty statements only."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tiledarray_amd",
                    "csrc")


def asm_texts(source):
    """The instruction text of every inline assembly statement."""
    for m in re.finditer(r'\basm\b(?:\s+volatile)?\s*\(\s*((?:"(?:[^"\\]|\\.)*"\s*)+)', source):
        yield "".join(re.findall(r'"((?:[^"\\]|\\.)*)"', m.group(1)))


def test_asm_texts_finds_instructions():
    assert list(asm_texts('asm("v_mov_b32 %0, %1" : "=v"(a)); asm volatile("" : "+v"(x));')) == [
        "v_mov_b32 %0, %1", ""]


def test_inline_assembly_holds_no_vector_instructions():
    files = sorted(glob.glob(os.path.join(CSRC, "*.h*")))
    assert files
    bad = [(os.path.basename(f), line) for f in files for text in asm_texts(open(f).read())
           for line in re.split(r"\\n|\\t|;", text)
           if line.strip() and line.split()[0] not in ("s_barrier", "s_waitcnt")]
    assert bad == []
