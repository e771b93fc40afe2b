"""Direct-to-LDS loads written in inline assembly: m0 is written by the scalar unit, and the vector memory instruction that reads it
needs one wait state behind that write. The compiler does not see into the text, so the text has to hold it."""
import glob
import os
import re

SOURCES = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "csrc")
INSTRUCTION = re.compile(r'"((?:[^"\\]|\\.)*)"')


def test_m0_is_followed_by_a_wait_state():
    seen = 0
    for path in sorted(glob.glob(os.path.join(SOURCES, "**", "*.h*"), recursive=True)):
        for text in INSTRUCTION.findall(open(path).read()):
            steps = [s.strip() for s in re.split(r"\\n|;", text.replace("\\t", " "))]
            for i, s in enumerate(steps):
                if re.match(r"s_\w+ +m0\b", s):
                    seen += 1
                    assert i + 1 < len(steps) and re.match(r"s_nop\b", steps[i + 1]), (path, text)
    assert seen > 0


def test_attention_opts_into_large_lds_on_every_device():
    """A kernel with more than 64 KB of dynamic LDS is opted in once on every device, not once a process: the second GPU of a process
    could not launch it. (One GPU cannot show that; a flag of the process can be seen in the source.)"""
    text = open(os.path.join(SOURCES, "kernels", "flash_attn.hip")).read()
    assert "set_lds_limit(" in text and not re.search(r"static\s+bool\s+\w+\s*=", text)
    # the opt-ins stand where the device is looked at, and nowhere else
    guarded = "".join(re.findall(r"on_each_device\(\w+, \[&\] \{(.*?)\n  \}\);", text, re.S))
    assert guarded.count("set_lds_limit(") == text.count("set_lds_limit(") - text.count("void set_lds_limit(")
