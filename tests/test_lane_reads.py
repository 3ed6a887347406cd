"""Values of other lanes (csrc/*.hip, csrc/*.h): what __builtin_amdgcn_readlane reads is a value that every lane has formed.

The lane that is read may be switched off where the read stands (behind a divergent branch). A value that was formed where all lanes are on
is in its register all the same; one that the read's own argument computes is not formed in that lane at all."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "comfyui_amd", "csrc")


def arguments(text, at):
    """The arguments of the call whose opening bracket is text[at]."""
    out, depth, start = [], 0, at + 1
    for i in range(at, len(text)):
        if text[i] in "([{":
            depth += 1
        elif text[i] in ")]}":
            depth -= 1
            if depth == 0:
                return out + [text[start:i].strip()]
        elif text[i] == "," and depth == 1:
            out.append(text[start:i].strip())
            start = i + 1


def test_no_lane_is_read_of_a_value_formed_for_the_read():
    seen = 0
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))):
        text = re.sub(r"//[^\n]*", "", open(path).read())
        for m in re.finditer(r"__builtin_amdgcn_readlane\(", text):
            value = arguments(text, m.end() - 1)[0]
            value = re.sub(r"^__float_as_uint\((.*)\)$", r"\1", value)   # the same register
            assert re.fullmatch(r"\w+(\.\w+)*", value), (os.path.basename(path), value)
            seen += 1
    assert seen >= 10
