"""Device memory is cleared on the stream that uses it.  Every context works on a non-blocking stream,
which nothing orders behind the null stream: a hipMemset on that may run after the kernels that rely
on it, or clear what they wrote.  hipMemsetAsync would be ordered, but its nodes in a captured graph
are not relied on here; clears are kernels."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "electron-phonon-hmc_amd", "csrc")


def test_clears_are_kernels_on_the_contexts_stream():
    files = glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))
    assert len(files) > 10
    found = []
    for path in sorted(files):
        with open(path) as f:
            for no, line in enumerate(f, 1):
                if re.search(r"\bhipMemset\w*\s*\(", line.split("//")[0]):
                    found.append("%s:%d %s" % (os.path.basename(path), no, line.strip()))
    assert not found, found
