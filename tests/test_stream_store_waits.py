"""Wait states around the inline-assembly stores, which the compiler's hazard pass does not see."""

import importlib
import os
import subprocess

import pytest

PROBE = """
#include "{csrc}/rlk_tile_epilogue.hpp"

__global__ void probe(const rlk::u32x4_t* a, float* out)
{{
    rlk::f32x4_t acc[8][1];
    for (int i = 0; i < 8; ++i) acc[i][0] = rlk::f32x4_t{{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i][0] = rlk::Bf16::mfma(a[threadIdx.x], a[threadIdx.x + 64 * i], acc[i][0]);
    rlk::settle_column(acc, 0);
#pragma unroll
    for (int i = 0; i < 8; ++i) rlk::stream_store(out + i * 256, threadIdx.x * 16, acc[i][0]);
}}
"""


@pytest.fixture(scope="module")
def builder():
    import rl_kernel_amd  # noqa: F401

    return importlib.import_module("rl_kernel_amd.build")


def test_stores_of_accumulators_keep_their_distances(builder, tmp_path):
    src, asm = tmp_path / "probe.hip", tmp_path / "probe.s"
    text = PROBE.format(csrc=builder.CSRC)
    src.write_text(text)
    res = subprocess.run([builder.hipcc(), *builder.HIPCC_FLAGS, "--cuda-device-only", "-S", str(src), "-o", str(asm),
                          f"-I{builder.CSRC}", f"-I{os.path.dirname(builder.HERE)}/include"],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    assert builder._check_stream_stores(str(asm), "probe") == 8


STORE = "\tglobal_store_dwordx4 v[0:1], v[8:11], off sc1 nt\n"
MFMA = "\tv_mfma_f32_16x16x32_bf16 {}, v[20:23], v[24:27], {}\n"


@pytest.mark.parametrize("asm,ok", [
    (STORE + "\ts_nop 1\n", True),
    (STORE + "\ts_nop 0\n", False),
    (STORE + "\tv_mov_b32_e32 v8, v9\n", False),
    (MFMA.format("v[8:11]", "v[8:11]") + "\ts_nop 11\n" + STORE + "\ts_nop 1\n", True),
    (MFMA.format("v[8:11]", "v[8:11]") + "\ts_nop 10\n" + STORE + "\ts_nop 1\n", False),
    (MFMA.format("v[12:15]", "v[12:15]") + STORE + "\ts_nop 1\n", True),
])
def test_the_build_refuses_short_distances(builder, tmp_path, asm, ok):
    path = tmp_path / "x.s"
    path.write_text(asm)
    if ok:
        assert builder._check_stream_stores(str(path), "x") == 1
    else:
        with pytest.raises(RuntimeError):
            builder._check_stream_stores(str(path), "x")
