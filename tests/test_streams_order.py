"""The key-stream kernel's LDS stages (csrc/fa_streams.h) are refilled by DMA
in inline assembly, which the compiler does not order behind an LDS read it has
issued: between a read of a stage and the next DMA into it the source itself
has to wait (``wait_lds``), whatever schedule a compiler picks."""
import os
import re

from custom_ops_amd import build

# what reads a stage, and the DMA that refills it
STAGES = {r"mk\.read\(": r"mk\.issue\(", r"a\.scores\(": r"issue_k\(", r"a\.pv\(": r"issue_v\("}


def kernel_body():
    with open(os.path.join(os.path.dirname(build.SRC), "fa_streams.h")) as f:
        text = f.read()
    body = re.sub(r"//[^\n]*", "", text[text.index("void fa_fwd_kernel_ks("):])
    for read, dma in STAGES.items():
        assert re.search(read, body) and re.search(dma, body)
    return body


def unordered(body):
    """Reads with no wait_lds() between them and the DMA that follows."""
    found = []
    for read, dma in STAGES.items():
        for m in re.finditer(read, body):
            nxt = re.compile(dma).search(body, m.end())
            if nxt and "wait_lds();" not in body[m.end():nxt.start()]:
                found.append(m.group())
    return found


def test_every_stage_read_is_waited_for_before_the_next_dma():
    assert unordered(kernel_body()) == []


def test_the_check_catches_a_missing_wait():
    waits = [m.start() for m in re.finditer(r"wait_lds\(\);", kernel_body())]
    assert len(waits) == 5   # the first follows the V stage's zero fill, a write
    for w in waits[1:]:
        body = kernel_body()
        assert unordered(body[:w] + body[w + len("wait_lds();"):]), w
