"""Device memory is cleared on a stream of the context that uses it: contexts'
streams are non-blocking, so the null stream is not ordered with them, and
hipMemset need not have finished when it returns."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fftcorr_amd",
                    "csrc")


def test_no_clearing_or_device_copy_on_the_null_stream():
    found = []
    for path in sorted(glob.glob(os.path.join(CSRC, "*"))):
        if os.path.isfile(path):
            text = open(path).read()
            for m in re.finditer(r"\bhipMemset(D\d+)?\s*\(|"
                                 r"\bhipMemcpy\s*\([^;]*hipMemcpyDeviceToDevice", text):
                found.append((os.path.basename(path), text.count("\n", 0, m.start()) + 1))
    assert not found, found
