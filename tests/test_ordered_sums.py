"""The ordered sums of the FP64 search (row_ordered_add, ordered_add), through
a probe of their own, against a serial sum on the host, bit for bit: every
count of lanes from 1 to 64, and the elements themselves as the accumulator
(the sum then must not take their register)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "native", "_ordered_probe.so")

pytestmark = pytest.mark.gpu


def probe(acc, v):
    if not os.path.exists(LIB):
        subprocess.run(["make", "-s", "-C", os.path.join(HERE, "..", "gpu-smina_amd"),
                        "../tests/native/_ordered_probe.so"], check=True)
    out = [np.zeros(64) for _ in range(3)] + [np.zeros(64, np.float32)]
    fn = C.CDLL(LIB).ordered_probe
    assert fn(*[x.ctypes.data_as(C.c_void_p) for x in (acc, v, *out)]) == 0
    return out


@pytest.mark.parametrize("seed", [1, 2])
def test_sums_equal_the_serial_sum(seed):
    rng = np.random.default_rng(seed)
    # magnitudes over 12 decades: every other order rounds differently
    acc, v = (rng.standard_normal(64) * 10.0 ** rng.uniform(-6, 6, 64) for _ in range(2))
    own, same, out, outf = probe(acc, v)
    for lane in range(64):
        for start, got in ((acc, own), (v, same)):
            s = start[lane]
            for x in v[lane // 16 * 16: lane // 16 * 16 + 16]:
                s = s + x
            assert got[lane] == s, (lane, got is same)
    for cnt in range(1, 65):
        s, sf = acc[0], np.float32(acc[0])
        for x in v[:cnt]:
            s, sf = s + x, sf + np.float32(x)
        assert out[cnt - 1] == s and outf[cnt - 1] == sf, cnt
