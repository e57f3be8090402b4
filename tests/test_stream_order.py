"""Device memory is filled on the stream that uses it.  The library's streams
do not wait for the default stream, and a fill without a stream need not have
ended when its call returns: kernels of the other stream could read the
memory before."""
import os
import re

import unifiedparticleframeworkcuda_amd as upf

CSRC = os.path.join(os.path.dirname(upf.__file__), "csrc")


def test_fills_name_their_stream():
    fills = 0
    for name in sorted(os.listdir(CSRC)):
        text = open(os.path.join(CSRC, name)).read()
        assert not re.findall(r"\bhipMemset(?:D8|D16|D32)?\(", text), name
        fills += len(re.findall(r"\bhipMemsetAsync\(", text))
    assert fills > 0
