"""The hash map behind the whole-stage kernel's block lists takes any number of
keys: a block at a node of very many cells is found not to fit after all of
their cells were seen.  Compiled here as it is, without a device."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fvs2d_amd", "csrc")
MAIN = """
#include "local_map.hpp"
#include <cstdio>
#include <cstdlib>
#include <map>
int main(int, char **v) {
  fvs::LocalMap m;
  for (int pass = 0; pass < 3; ++pass) {
    std::map<unsigned, int> ref;
    const int n = pass == 1 ? 100 : atoi(v[1]);
    for (int k = 0; k < n; ++k) {
      const unsigned key = unsigned(k % (n - n / 8)) * unsigned(atoi(v[2])) | unsigned(k % 15) << 27;
      bool fresh;
      int &x = m.at(key, fresh);
      if (fresh != (ref.count(key) == 0)) return 1;
      if (fresh) x = ref[key] = k;
      if (x != ref[key]) return 2;
    }
    if (m.size() != ref.size()) return 3;
    for (auto &e : ref) {
      bool fresh;
      if (m.at(e.first, fresh) != e.second || fresh) return 4;
    }
    m.clear();
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("map")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "main")],
                   check=True)
    return str(d / "main")


@pytest.mark.parametrize("stride", [1, 64, 256, 4096])
@pytest.mark.parametrize("keys", [20, 128, 256, 8192, 9000, 30000])
def test_any_number_of_keys(program, keys, stride):
    assert subprocess.run([program, str(keys), str(stride)], timeout=20).returncode == 0
