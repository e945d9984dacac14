"""The library issues nothing on the null stream: a null-stream call fails
while any thread of the process captures a graph, which every launch of a
new kernel variant does."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "imagevis3d_amd", "csrc")


def code_of(path):
    with open(path) as f:
        s = f.read()
    s = re.sub(r"/\*.*?\*/", "", s, flags=re.S)
    return re.sub(r"//[^\n]*", "", s)


def test_no_call_without_a_stream():
    bad = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*"))):
        code = code_of(path)
        # blocking copies and fills, streams that order themselves with the
        # null stream, launches without a stream or with a null one
        for pat in (r"\bhipMemcpy(2D|3D)?\s*\(", r"\bhipMemset(D8|D16|D32|2D)?\s*\(", r"\bhipMemcpy(To|From)Symbol\s*\(",
                    r"\bhipStreamCreate\s*\(", r"\bhipDeviceSynchronize\s*\(",
                    r"\blaunch_\w+\s*\([^;{]*,\s*(nullptr|0)\s*\)\s*;"):
            bad += [f"{os.path.basename(path)}: {m.group(0)}" for m in re.finditer(pat, code)]
        for m in re.finditer(r"<<<(.*?)>>>", code, flags=re.S):
            if not re.search(r"\bstream_?$", m.group(1).strip()):
                bad.append(f"{os.path.basename(path)}: {m.group(0)}")
    assert not bad, bad
