"""No status of a launch or of a runtime call is dropped: every source
compiles (host pass, nothing generated) with the package's flags, which make
an unused hipError_t an error."""
import concurrent.futures as cf
import os
import subprocess

import pytest

from pdl_amd import build as B

UNITS = {src: extra for src, name, extra in reversed(B.units())}   # one unit of each source


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="no hipcc")
def test_every_status_is_used():
    assert "-Werror=unused-value" in B.FLAGS

    def check(src):
        r = subprocess.run([B.HIPCC] + B.FLAGS + UNITS[src] + ["--cuda-host-only", "-fsyntax-only",
                                                              os.path.join(B.CSRC, src)],
                           capture_output=True, text=True)
        return "" if r.returncode == 0 else src + "\n" + r.stderr[-2000:]

    with cf.ThreadPoolExecutor(4) as ex:
        failed = [x for x in ex.map(check, sorted(UNITS)) if x]
    assert not failed, "\n".join(failed)
