"""The order in which singular values are sorted (tenes_amd/csrc/rank.hpp),
compiled for the host: ranks of any values, NaN among them, are a permutation."""
import ctypes
import itertools
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "tenes_amd" / "csrc"


@pytest.fixture(scope="module")
def before(tmp_path_factory):
    d = tmp_path_factory.mktemp("rank")
    (d / "r.cpp").write_text('#include "rank.hpp"\nextern "C" int before(double u, int k, double v, int j) '
                             "{ return tn::ranks_before(tn::rank_key(u), k, tn::rank_key(v), j); }\n")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", str(d / "r.cpp"), "-o", str(d / "r.so")],
                   check=True)
    f = ctypes.CDLL(str(d / "r.so")).before
    f.argtypes = [ctypes.c_double, ctypes.c_int, ctypes.c_double, ctypes.c_int]
    return f


def test_ranks_are_a_permutation(before):
    """As sort_desc_kernel counts them: rank j = number of values before it."""
    for values in itertools.product([np.nan, np.inf, 2.0, 0.0, -0.0], repeat=4):
        n = len(values)
        rank = [sum(before(values[k], k, values[j], j) for k in range(n)) for j in range(n)]
        assert sorted(rank) == list(range(n)), (values, rank)
        out = np.empty(n)
        out[rank] = values
        numbers = out[~np.isnan(out)]
        assert np.all(np.isnan(out[len(numbers):])) and np.all(numbers[:-1] >= numbers[1:])
        for a, b in itertools.combinations(range(n), 2):  # equal values keep their order
            if values[a] == values[b] or (np.isnan(values[a]) and np.isnan(values[b])):
                assert rank[a] < rank[b]
