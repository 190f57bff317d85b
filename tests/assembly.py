"""The instructions that the compiler makes of this package's kernels, for tests of what no result shows."""

import functools
import re
import subprocess
import tempfile

from halite_amd.kernels import library


@functools.lru_cache(maxsize=None)
def kernels(source):
    """The lines of every kernel of a file under ``csrc``, by its name in the library."""
    with tempfile.TemporaryDirectory() as folder:
        out = f"{folder}/{source}.s"
        subprocess.run([library._hipcc(), *library.HIPCC_FLAGS, "--offload-device-only", "-S", "-I", library.CSRC, f"{library.CSRC}/{source}", "-o", out],
                       check=True, capture_output=True)
        with open(out) as f:
            text = f.read()
    found, lines = {}, None
    for line in text.splitlines():
        if m := re.match(r"(_Z\w+):", line):
            lines = found[m[1]] = []
        elif line.startswith("\t.section"):
            lines = None
        elif lines is not None:
            lines.append(line.split(";")[0].strip())
    return found
