"""Which transforms have a paired kernel, read from the lists the kernels are
built from, so that a test for the other path can say that it takes it."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "baandi_amd", "csrc")


def _entries(source, macro):
    with open(os.path.join(CSRC, source)) as f:
        text = f.read().replace("\\\n", " ")
    body = re.search(r"#define %s\(X\)(.*)" % macro, text).group(1)
    found = [tuple(int(v) for v in e.split(",")) for e in re.findall(r"X\(([\d, ]+)\)", body)]
    assert found, macro
    return found


def paired_planes():
    """(n1, n2) of plane_kernels.hpp."""
    return {(split * ya * yb, a * b) for split, ya, yb, a, b in _entries("plane_kernels.hpp", "BD_PLANES")}


def paired_lengths():
    """x lengths of stick.hip."""
    return {a * b for a, b in _entries("stick.hip", "BD_LINES")}


def paired_cubes():
    """Axis lengths of kpair.hip."""
    return {a * b for a, b in _entries("kpair.hip", "BD_CUBES")}
