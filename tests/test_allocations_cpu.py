"""Every device allocation of the library goes through dev_malloc, which frees
the buffers kept for later calls and tries again when memory runs out."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hpcscan_amd", "csrc")


def test_device_memory_is_allocated_in_one_place():
    calls = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*"))):
        with open(path) as f:
            text = re.sub(r"//[^\n]*|/\*.*?\*/|\"[^\"\n]*\"", "", f.read(), flags=re.S)
        inside = re.search(r"\nhipError_t dev_malloc\([^;{]*\)\n\{.*?\n}\n", text, flags=re.S)
        if inside:
            text = text.replace(inside.group(0), "")
            calls.append("dev_malloc")
        calls += [f"{os.path.basename(path)}: {m}" for m in re.findall(r"\bhip(?:Ext)?Malloc\w*", text)]
    assert calls == ["dev_malloc"]
