"""How the EHSS and surrogate kernels spread a cloud: the rules themselves (host
code), at the sizes where a round of wavefronts fills."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "icarion_amd", "csrc")
SHIM = """
#include "launch_rules.hpp"
extern "C" uint32_t ehss(uint32_t n, uint32_t w) { return icarion::ehss_ions_per_wave(n, w); }
extern "C" uint32_t ehss_waves(int i, int a, int x) { return icarion::ehss_waves_per_simd(i, a, x); }
extern "C" uint32_t surrogate(uint32_t n) { return icarion::surrogate_ions_per_wave(n); }
extern "C" int large(uint32_t n) { return icarion::surrogate_large(n); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, lib = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(src), "-o", str(lib)], check=True)
    so = ctypes.CDLL(str(lib))
    so.ehss.restype = so.surrogate.restype = so.ehss_waves.restype = ctypes.c_uint32
    so.ehss.argtypes, so.surrogate.argtypes, so.large.argtypes = [ctypes.c_uint32] * 2, [ctypes.c_uint32], [ctypes.c_uint32]
    return so


SIZES = [0, 1, 1023, 1024, 1025, 2048, 2049, 43008, 45057, 64512, 64513, 65535, 65536, 65537, 129025, 131071, 131072,
         131073, 262144, 262145, 1_000_000, 2**32 - 1]


@pytest.mark.parametrize("n", SIZES)
def test_surrogate_instantiation_follows_the_ion_count(rules, n):
    """The four-wavefront instantiation runs above 131,072 ions and nowhere below,
    where one or two wavefronts per SIMD gain from the registers instead."""
    assert bool(rules.large(n)) == (n > 131072)
    g = rules.surrogate(n)
    assert 1 <= g <= 64
    waves = -(-n // g)
    assert g == 64 or waves <= 2048
    if n > 131072:
        assert g == 64


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("per_simd", [1, 2])
def test_ehss_rounds_fill_the_chip_as_the_kernel_holds_it(rules, n, per_simd):
    """No more wavefronts than the full rounds hold, and no round more than full
    wavefronts would take."""
    g = rules.ehss(n, per_simd)
    assert 1 <= g <= 64
    slots = 1024 * per_simd
    rounds = -(-n // (64 * slots))
    assert -(-n // g) <= max(rounds, 1) * slots


def test_ehss_wavefronts_per_simd(rules):
    assert [rules.ehss_waves(i, a, x) for i, a, x in
            ((0, 0, 0), (1, 0, 0), (0, 1, 0), (1, 1, 0), (0, 0, 1), (1, 0, 1))] == [2, 2, 1, 2, 1, 1]
