"""Wait states around inline assembly, which the compiler's hazard pass does not see."""

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


def device_code(builder, tmp_path, text):
    src, asm = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(text.format(csrc=builder.CSRC))
    res = subprocess.run([builder.hipcc(), *builder.HIPCC_FLAGS, "--cuda-device-only", "-S", str(src), "-o", str(asm),
                          f"-I{builder.CSRC}", f"-I{os.path.dirname(builder.HERE)}/include"],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    return str(asm)


def test_stores_of_accumulators_keep_their_distances(builder, tmp_path):
    assert builder._check_stream_stores(device_code(builder, tmp_path, PROBE), "probe") == 8


LOAD_PROBE = """
#include "{csrc}/rlk_gemm.hpp"

__global__ __launch_bounds__(512) void probe(const uint16_t* a, float* out)
{{
    __shared__ __attribute__((aligned(16))) char tile[32768];
    rlk::DtlIO<false, 256, 64> io;
    io.init(rlk::Operand{{a, 64, 256}}, 64);
    for (int p = 0; p < decltype(io)::kPasses; ++p) io.load_one(0, tile, p);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    out[threadIdx.x] = reinterpret_cast<float*>(tile)[threadIdx.x];
}}
"""


def test_loads_to_lds_wait_for_their_destination(builder, tmp_path):
    assert builder._check_m0_loads(device_code(builder, tmp_path, LOAD_PROBE), "probe") == 4
    short = tmp_path / "short.s"
    short.write_text("\ts_mov_b32 m0, s4\n\tglobal_load_lds_dwordx4 v2, s[0:1]\n")
    with pytest.raises(RuntimeError):
        builder._check_m0_loads(str(short), "short")


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


@pytest.mark.parametrize("name,ok", [("_ZN3rlk21linear_logp_dw_kernelI4Bf16Li64EEvT_", False),
                                     ("_ZN3rlk24linear_logp_grads_kernelI4Bf16Li64ELb1EEvT_", True)])
def test_the_build_refuses_streaming_stores_in_the_unchained_kernel(builder, tmp_path, name, ok):
    path = tmp_path / "x.s"
    path.write_text(f"{name}:  ; @{name}\n" + STORE + "\ts_nop 1\n\ts_endpgm\n")
    if ok:
        assert builder._check_cached_stores(str(path), "x") == 0
    else:
        with pytest.raises(RuntimeError):
            builder._check_cached_stores(str(path), "x")
