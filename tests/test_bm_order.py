"""Block matching's paired form keeps the reference search's candidate list
over the tile that the search reads.  The list's positions are integers and
depend on no distance, the tile's samples are floats: under the type-based
alias rules only a wavefront fence between the two keeps a compiler from
storing positions over samples that other lanes have yet to read.  No
present compiler output shows it, so the fence is looked for where it has to
stand: in the unoptimised device IR of every instantiation, between the
first sum of squared differences and the first selection."""
import os
import re
import subprocess

import pytest

from conftest import ROOT
from vbm3d_amd import build as B


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    out = tmp_path_factory.mktemp("ir") / "kernels_bm.ll"
    subprocess.check_call([B.HIPCC, *B.FLAGS, "--offload-device-only", "-S", "-emit-llvm", "-Xclang",
                           "-disable-llvm-passes", "-o", str(out), os.path.join(ROOT, "vbm3d_amd", "csrc", "kernels_bm.hip")],
                          stderr=subprocess.DEVNULL)
    return re.findall(r"^define [^@]*@(_ZN2vb12_GLOBAL__N_16bm_one\w+)\(.*?^}", out.read_text(), re.S | re.M), \
        re.split(r"^(?=define )", out.read_text(), flags=re.M)


def test_reference_search_fences_its_list(functions):
    names, bodies = functions
    assert len(names) >= 30  # patch sizes 4..8, one and three channels, shapes, temporal form
    seen = 0
    for b in bodies:
        m = re.match(r"define [^@]*@(_ZN2vb12_GLOBAL__N_16bm_one\w+)\(", b)
        if not m:
            continue
        calls = re.findall(r"call [^@]*@(\w+)\(", b)
        ssd = next(i for i, c in enumerate(calls) if re.search(r"bm_one\w+ENKUlPKfiifjE_cl", c))
        sel = next(i for i, c in enumerate(calls) if "wave_select" in c)
        fences = sum("wave_sync" in c for c in calls[ssd + 1:sel])
        # one between the tile's reads and the list's stores, one between those and the selection
        assert fences == 2, (m.group(1), fences)
        seen += 1
    assert seen == len(names)
