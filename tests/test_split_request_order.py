"""The order in which the kernel of few q-blocks asks for its tiles at head size 128.  Its waits count requests (all but the newest
2 * DT have landed), so the DMA of K has to stay in front of the loads of V whatever the scheduler prefers: looked up in the
assembly of csrc/attn_sparse_split.hip, as it is built and under a scheduling strategy that moves loads further."""
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor
from itertools import groupby
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parent.parent / "paroatten_amd"


def _build_module():
    import importlib.util
    spec = importlib.util.spec_from_file_location("_paro_build_order", PKG / "build.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


FORMS = {"as_built": (), "max_ilp": ("-mllvm", "-amdgpu-sched-strategy=max-ilp")}


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    build, where = _build_module(), tmp_path_factory.mktemp("asm")
    try:
        cc = build.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")

    def compile_to(form):
        out = where / (form + ".s")
        r = subprocess.run([cc, *build.FLAGS, *FORMS[form], "-S", "--offload-device-only", str(PKG / "csrc" / "attn_sparse_split.hip"),
                            "-o", str(out)], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        return out.read_text()
    with ThreadPoolExecutor(2) as ex:
        return dict(zip(FORMS, ex.map(compile_to, FORMS)))


@pytest.mark.parametrize("form", FORMS)
def test_k_is_requested_in_front_of_v(assembly, form):
    kernels = {}
    name = None
    for line in assembly[form].splitlines():
        m = re.match(r"(_ZN4paro24attn_sparse_split_kernelILi128\w+):", line)
        if m:
            name = m.group(1)
            kernels[name] = ""
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name and line.strip().startswith("buffer_load"):
            kernels[name] += "K" if line.rstrip().endswith(" lds") else "v"
    assert len(kernels) == 24   # two types, log-sum-exp / true / fast exponentials, two widths, Q in 8 and 16 bits
    for name, loads in kernels.items():
        runs = [(c, len(list(g))) for c, g in groupby(loads)]
        # the first block's K in fragments, two tiles by DMA, V; then per round (two of them, one for each parity) one tile and its V
        assert runs == [("v", 8), ("K", 16), ("v", 8), ("K", 8), ("v", 8), ("K", 8), ("v", 8)], (name, runs)
