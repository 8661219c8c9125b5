"""When an FP16 inference deals its tiles by the device count (csrc/nrc_deal.hpp, host code), on 256 CUs
with two workgroups of four waves each."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WAVES = 2048


@pytest.fixture(scope="module")
def limits(tmp_path_factory):
    d = tmp_path_factory.mktemp("deal")
    src, so = d / "deal.cpp", d / "deal.so"
    src.write_text('#include "nrc_deal.hpp"\n'
                   'extern "C" void limits(unsigned tiles, unsigned waves, unsigned per_cu, unsigned *o) {\n'
                   '  const nrc::DealLimits l = nrc::infer_deal_limits(tiles, waves, per_cu);\n'
                   '  o[0] = l.split; o[1] = l.all; o[2] = l.some; }\n')
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "vknrc_amd", "csrc"), str(src), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))

    def get(tiles, waves=WAVES, per_cu=2):
        o = (C.c_uint32 * 3)()
        lib.limits(tiles, waves, per_cu, o)
        return tuple(o)
    return get


def by_count(limits, queries, count):
    """As infer_tiles (nrc_mfma.hpp) decides."""
    split, all_, some = limits(-(-queries // 64))
    t = -(-count // 64)
    return all_ != 0 and t <= (all_ if t > split else some)


# where the deal by the count took 1.03 to 1.17 of the time of the deal by the maximum
@pytest.mark.parametrize("queries,fraction", [(196608, f) for f in (0.999, 0.98, 0.95, 0.92, 0.88, 0.8)] + [
    (262144, 0.5), (262144, 0.4), (393216, 0.88), (393216, 0.5), (524288, 0.95), (524288, 0.92), (524288, 0.88)])
def test_dealt_by_the_maximum(limits, queries, fraction):
    assert not by_count(limits, queries, int(queries * fraction))


# where it took 0.14 to 0.95
@pytest.mark.parametrize("queries,fraction", [(140000, 0.92), (140000, 0.6), (140000, 0.1), (196608, 0.6), (196608, 0.25), (262144, 0.25),
                                              (393216, 0.7), (393216, 0.6), (393216, 0.25), (524288, 0.7), (524288, 0.26), (524288, 0.25),
                                              (720000, 0.6), (921600, 0.92), (921600, 700001 / 921600), (921600, 0.4), (921600, 0.01),
                                              (2073600, 0.88), (2073600, 0.25), (2073600, 0.01)])
def test_dealt_by_the_count(limits, queries, fraction):
    assert by_count(limits, queries, int(queries * fraction))


def test_limits_of_any_launch(limits):
    for per_cu in range(1, 9):
        waves = 1024 * per_cu
        for tiles in (0, 1, waves - 1, waves, waves + 1, 3 * waves, 3 * waves + 5, (1 << 31) // 64):
            split, all_, some = limits(tiles, waves, per_cu)
            if tiles <= waves:
                assert all_ == 0  # one tile a wave at most either way
            else:
                assert 0 < some <= all_ and split < tiles and all_ < tiles + waves
    assert not by_count(limits, 64 * WAVES, 1) and by_count(limits, 64 * WAVES + 1, 1)
