"""The host code on a recording stand-in for the HIP runtime
(tests/host/fake_hip.hpp): the sizes, routes and orders of what a call
allocates and launches, at shapes and in situations that need no GPU."""
import pathlib
import re
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parent.parent
PKG = ROOT / "ltx-zml_amd"


@pytest.fixture(scope="session")
def host_paths(tmp_path_factory):
    exe = tmp_path_factory.mktemp("host") / "host_paths"
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-Wno-unused-result", "-rdynamic",
                    "-I/opt/rocm/include", f"-I{ROOT / 'include'}", f"-I{PKG / 'csrc'}", f"-I{PKG / 'csrc' / 'host'}",
                    str(ROOT / "tests" / "host" / "host_paths.cpp"), "-o", str(exe), str(PKG / "libltx_amd.so"),
                    f"-Wl,-rpath,{PKG}", "-Wl,--allow-shlib-undefined", "-pthread"], check=True)

    def run(*args):
        r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
        return r.stdout
    return run


@pytest.mark.parametrize("T,S", [(1024, 128), (65535, 128), (65536, 128), (262143, 77), (262144, 128), (64, 262144)])
def test_f32_block_planes_fit_their_room(host_paths, T, S):
    """Token counts on both sides of where the GEMM on planes stops taking the
    K = 16,384 projection (65,536) and the K = 4,096 ones (262,144)."""
    host_paths("f32_planes", T, S)


def test_f32_block_without_room_for_planes(host_paths):
    host_paths("f32_workspace")


@pytest.mark.parametrize("scratch", ["planes", "vt"])
def test_operator_scratch_is_ordered(host_paths, scratch):
    """Calls that share a context's operator scratch (mode F32's planes, the
    attention's padded V^T) follow each other: on one stream handle, on two, and
    behind a call that failed between its launches."""
    host_paths(f"scratch_order_{scratch}")


def test_operator_scratch_grows_beside_a_capture(host_paths):
    host_paths("scratch_capture")


def test_operator_scratch_without_memory(host_paths):
    host_paths("scratch_memory")


@pytest.mark.parametrize("M,N,K", [(1024, 12288, 4096), (1, 128, 128), (300, 256, 4096), (28672, 4096, 16384),
                                   (5377, 4096, 16384), (65535, 128, 16384), (200000, 128, 4096), (129, 128, 32768)])
def test_f32_linear_planes_are_bounded(host_paths, M, N, K):
    host_paths("planes_bound", M, N, K)


@pytest.mark.parametrize("captured", [0, 1])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("T,S", [(250, 40), (256, 64), (1024, 77), (2970, 128), (2970, 100), (4100, 1), (8200, 300)])
def test_stages_of_v_stay_in_the_workspace(host_paths, T, S, mode, captured):
    """Whole and ragged token counts on every schedule of the second stream, int8
    and (mode 1) unquantised weights."""
    host_paths("stage_v", T, S, mode, captured)


def test_noalloc_f32_calls_are_independent(host_paths):
    host_paths("noalloc_f32")


@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (300, 256, 4096), (3000, 128, 4096), (28672, 4096, 16384),
                                   (1000, 4096, 32768), (129, 128, 32768)])
def test_noalloc_f32_planes_fit_the_array(host_paths, M, N, K):
    host_paths("planes_bound_noalloc", M, N, K)


def test_attention_with_misaligned_keys_stays_any_length(host_paths):
    """Ragged key counts with K off a 16-byte boundary: not for 16-byte LDS DMA."""
    host_paths("attn_misaligned")


def test_linear_allocates_nothing_once_warmed(host_paths):
    host_paths("linear_warmed")


def test_attention_pads_where_it_pays(host_paths):
    """(queries, keys) on both sides of each line of the padding rule: the calls
    measured faster on the any-length kernel stay on it."""
    any_length = [(200, 16), (1000, 255), (2048, 264), (2049, 72), (2100, 77), (2100, 130), (2304, 712), (2305, 264),
                  (2500, 200), (3000, 50), (3000, 264), (4000, 200), (4096, 63), (4097, 200), (4200, 72), (5000, 50)]
    padded = [(200, 300), (1025, 450), (2100, 250), (2304, 776), (2305, 65), (2500, 328), (3000, 130), (3500, 264),
              (4096, 264), (4097, 65), (4200, 264), (4353, 72), (5000, 200), (6145, 1), (8200, 16)]
    out = host_paths("attn_padded", *(n for pair in any_length + padded for n in pair)).split()[:-1]
    assert [p for p, o in zip(any_length + padded, out) if (o == "1") != (p in padded)] == []


def test_gemm_tile_heights(host_paths):
    """(M, N, K, f16 scales) on both sides of each line of the rule for tiles of
    192 rows: the calls measured faster on 256 rows stay there."""
    r256 = [(3500, 16384, 4096, 0), (3500, 16384, 4096, 1), (15360, 4096, 4096, 1), (13000, 4096, 16384, 1),
            (17000, 4096, 16384, 0), (21000, 4096, 16384, 0), (15000, 12288, 4096, 1), (28672, 4096, 4096, 1),
            (4095, 4096, 4096, 1), (2970, 16384, 4096, 0)]
    r192 = [(4100, 4096, 4096, 0), (9216, 4096, 16384, 1), (2970, 12288, 4096, 0), (5400, 12288, 4096, 1),
            (16500, 8192, 4096, 1), (18432, 4096, 4096, 0), (2100, 4096, 4096, 0), (2500, 4096, 4096, 0)]
    out = host_paths("tile_rows", *(n for shape in r256 + r192 for n in shape)).split()[:-1]
    assert [s for s, o in zip(r256 + r192, out) if (o == "1") != (s in r192)] == []


def test_gate_logits_fit_beside_the_16_bit_gemm(tmp_path):
    """The gate logits run on the second stream beside the 16-bit-weight GEMM
    (unquantised blocks up to 2,048 tokens): a workgroup of theirs has to fit
    what that GEMM leaves of a CU. 160 KB of LDS in pieces of 1,280 bytes; 512
    registers a lane of a SIMD, in eights, for two waves of each."""
    bundle = PKG / "_build" / "k_gemm.hsaco"
    llvm = pathlib.Path("/opt/rocm/llvm/bin")
    if not bundle.exists() or not (llvm / "llvm-readelf").exists():
        pytest.skip("no built code object, or no LLVM tools to read it")
    co = tmp_path / "k_gemm.co"
    subprocess.run([llvm / "clang-offload-bundler", "--type=o", "--unbundle",
                    "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={bundle}", f"--output={co}"], check=True)
    notes = subprocess.run([llvm / "llvm-readelf", "--notes", co], capture_output=True, text=True, check=True).stdout
    kernels = {}
    for entry in re.split(r"\n  - \.agpr_count", notes)[1:]:
        get = lambda key: re.search(rf"\.{key}:\s+(\S+)", entry)[1]  # noqa: E731
        kernels[get("name")] = (int(get("group_segment_fixed_size")), int(get("vgpr_count")))
    for dt in ("f16", "bf16"):
        gate = kernels[f"ltx_gate_{dt}"]
        for gemm in (kernels[f"ltx_gemm_w16dma_{dt}_qkv"], kernels[f"ltx_gemm_w16dma_{dt}_store"]):
            assert sum(-(-lds // 1280) * 1280 for lds, _ in (gate, gemm)) <= 160 * 1024
            assert sum(2 * -(-regs // 8) * 8 for _, regs in (gate, gemm)) <= 512
