"""What the compiler gave the hot kernels, read from the built library's own code objects: no scratch memory in kernels whose inner
loops would pay for every spilled register.  No GPU is needed."""
import os
import re
import subprocess

import pytest

from born_amd import _capi

LLVM = "/opt/rocm/llvm/bin"

#: kernel -> a pattern of its mangled names
HOT = {"sampling without a top-k cut": r"nucleus_row_kernelILi\d+E", "the same, a row's own settings": r"nucleus_row_rows_kernelILi\d+E",
       "top-k sampling": r"topk_row(_rows)?_kernelILi\d+E", "token log-probabilities": "token_logprob", "verification": "spec_",
       "softmax": "softmax_", "large products, weights of a linear layer": r"gemm_split_kernelILb1E", "fp32 products": r"gemm_f32_",
       "few rows of a linear layer": r"gemm_rows_kernel", "small products": r"gemm_small_kernel", "rows in parts: the sweeps": r"nucleus_parts_(max|masses|gather)", "the left operand's parts": r"gemm_split_pack"}

#: kernels that keep some registers in scratch, outside their inner loops -> the most bytes a lane
SOME = {"rows of every kind in one launch": (r"any_row_kernel", 276), "rows in parts: the draw": (r"nucleus_parts_draw", 8),
        "large products, [K,N] weights": (r"gemm_split_kernelILb0E", 84)}


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Mangled name -> its metadata (numbers)."""
    d = tmp_path_factory.mktemp("objects")
    fat = str(d / "fatbin")
    subprocess.check_call([LLVM + "/llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, _capi.LIB_PATH, str(d / "lib.so")])
    data, got = open(fat, "rb").read(), {}
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__|CCOB", data)]
    for i, at in enumerate(starts):                            # one bundle a source file
        part, obj = str(d / f"{i}.bundle"), str(d / f"{i}.o")
        open(part, "wb").write(data[at:(starts + [len(data)])[i + 1]])
        subprocess.check_call([LLVM + "/clang-offload-bundler", "--unbundle", "--type=o", "--input=" + part, "--output=" + obj,
                               "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"])
        notes = subprocess.check_output([LLVM + "/llvm-readelf", "--notes", obj], text=True)
        for block in re.split(r"\n  - \.a", notes)[1:]:
            name = re.search(r"\n    \.name: +(\S+)", block).group(1)
            got[name] = {k: int(v) for k, v in re.findall(r"\n    \.(\w+): +(\d+)\b", block)}
    return got


@pytest.mark.parametrize("kernel", HOT)
def test_no_scratch(kernels, kernel):
    of = {n: k for n, k in kernels.items() if re.search(HOT[kernel], n)}
    assert of, "no such kernel in the library"
    bad = {n: k["private_segment_fixed_size"] for n, k in of.items() if k["private_segment_fixed_size"] or k["vgpr_spill_count"]}
    assert not bad, bad


@pytest.mark.parametrize("kernel", SOME)
def test_no_more_scratch(kernels, kernel):
    of = {n: k["private_segment_fixed_size"] for n, k in kernels.items() if re.search(SOME[kernel][0], n)}
    assert of and max(of.values()) <= SOME[kernel][1], of
