"""A partial of the persistent kernel is complete before its tag can be seen: in
the code compiled for the GPU the words are stored, the wave waits for them and
its lanes meet, and only then the tag is stored. (On the CPU: nothing runs.)"""
import importlib.util
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "gw-model_amd")

SOURCE = """
#include "gw_kernels.h"
__global__ void k_post(gw::Partial *p, const uint64_t *w, int64_t n)
{
    const int t = threadIdx.x;
    gw::post_partial(*p, t, t < gw::PW_N ? w[t] : 0, n);
}
"""


def _build_ext():
    spec = importlib.util.spec_from_file_location("gw_build_ext", os.path.join(PKG, "build_ext.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_the_tag_of_a_partial_is_stored_after_its_words(tmp_path):
    be = _build_ext()
    if not os.path.exists(be.HIPCC):
        pytest.skip("no hipcc")
    src, out = tmp_path / "post.hip", tmp_path / "post.s"
    src.write_text(SOURCE)
    flags = [f for f in be.HIP_FLAGS if f != "-shared"]
    subprocess.run([be.HIPCC, *flags, "--cuda-device-only", "-S", f"-I{os.path.join(PKG, 'csrc')}", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    body = out.read_text().split("k_post", 1)[1].split("s_endpgm", 1)[0]
    order = re.findall(r"^\s*(global_store|flat_store|s_waitcnt vmcnt\(0\)|; wave barrier)", body, flags=re.M)
    stores = [i for i, x in enumerate(order) if x.endswith("_store")]
    assert len(stores) == 2, order
    between = order[stores[0] + 1:stores[1]]
    assert "; wave barrier" in between, order
    assert "s_waitcnt vmcnt(0)" in between[:between.index("; wave barrier")], order
