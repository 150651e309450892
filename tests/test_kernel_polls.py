"""Device loops whose lanes wait for one another: every one ends its pass where a successful poll and one
in vain meet (poll_end), or the compiler may give the vain polls a loop of their own, in which a
wavefront waits for its own lanes for ever."""
import os
import re

SOURCE = os.path.join(os.path.dirname(__file__), "..", "pypybox2d_amd", "csrc", "b2g_engine.hip")


def _block(text, start):
    depth = 0
    for i in range(text.index("{", start), len(text)):
        depth += (text[i] == "{") - (text[i] == "}")
        if depth == 0:
            return text[start:i]
    raise AssertionError("unbalanced braces")


def test_every_polling_loop_ends_its_pass_in_one_place():
    text = open(SOURCE).read()
    loops = [_block(text, m.start()) for m in re.finditer(r"while \(wave_any\([^\n]*poll < ", text)]
    assert len(loops) == 3  # the island search's levels, the group solver's velocities and positions
    for loop in loops:
        solved = loop.rindex("if ((") if "if ((" in loop else loop.rindex("if (todo")
        end = solved + len(_block(loop, solved))
        assert re.match(r"\}\s*poll_end\(", loop[end:]), loop[:200]
