"""The kernels that bench.py names in its rooflines exist in the built library (no GPU)."""
import re
from pathlib import Path

from dlcompiler_amd.build import kernel_resources


def test_named_kernels_are_built():
    text = (Path(__file__).resolve().parents[1] / "bench.py").read_text()
    named = set()
    for value in re.findall(r'"kernel": "([^"]*)"', text) + re.findall(r'msk?, "(\w+)[^"]*"', text):
        named |= {n for n in re.findall(r"\w+", value) if n.endswith("_kernel") or n.endswith("_vec16")}
    built = " ".join(kernel_resources())
    assert len(named) > 5
    assert not [n for n in named if n not in built]
