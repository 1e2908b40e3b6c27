"""The lengths of the two-launch attempts and of the grouped convolutions are
split over translation units: each even 2^a 3^b 5^c 7^d from 48 to 512 in
exactly one of them."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fastisostasy_amd", "csrc")


def lengths():
    def smooth(n):
        for p in (2, 3, 5, 7):
            while n % p == 0:
                n //= p
        return n == 1
    return [n for n in range(48, 513, 2) if smooth(n)]


@pytest.mark.parametrize("files,call", [("rhs_turn*.hip", "turn_lookup"), ("conv_mix*.hip", "conv_mix_lookup")])
def test_every_length_once(files, call):
    got = []
    for path in glob.glob(os.path.join(CSRC, files)):
        with open(path) as f:
            got += [int(v) for m in re.findall(call + r"<([^>]*)>", f.read()) for v in m.split(",")]
    assert sorted(got) == lengths()
