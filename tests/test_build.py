"""The in-tree native libraries build for gfx950 and load on a CPU-only host (catches
undefined symbols / missing registrations before a GPU box ever sees them)."""
import re
import struct
import subprocess
import types
from pathlib import Path

import pytest
import torch

from agentic_traffic_testing_amd.ops import build

EXPECTED_OPS = {
    "rms_norm", "fused_add_rms_norm", "silu_and_mul", "embed", "stream_read", "rope_cache",
    "attention_prefill",
    "attention_decode", "attention_decode_v2", "sample", "skinny_gemm", "fused_qkv_rope",
    "fused_gate_up_silu", "fused_lm_head_sample", "sample_finalize", "skinny_variant",
    "ar_buffer_bytes", "ar_alloc", "ar_free", "ar_handle", "ar_open", "ar_close", "ar_error",
    "ar_run",
}


def test_kernel_library_loads_and_registers_all_ops():
    so = build.build_kernels()
    torch.ops.load_library(str(so))
    for name in EXPECTED_OPS:
        assert hasattr(torch.ops.atta, name), name
        getattr(torch.ops.atta, name).default  # schema registered
    # host-only helper callable without a GPU
    assert torch.ops.atta.ar_buffer_bytes(1024, 2) == 64 * 1024 + 2 * 8 * 1024 * 2


def test_runtime_extension_loads():
    from agentic_traffic_testing_amd.runtime import BlockManager, ShmChannel

    bm = BlockManager(8, 16, True)
    assert bm.num_free_blocks() == 8
    assert ShmChannel is not None


def test_embed_cpu_fallback_honours_lookahead_flag():
    from agentic_traffic_testing_amd import ops

    table = torch.randn(50, 16)
    ids = torch.tensor([1, 2, 3], dtype=torch.int32)
    prev = torch.tensor([7, 8, 9, 10], dtype=torch.int64)
    assert torch.equal(ops.embed(table, ids), table[[1, 2, 3]])
    assert torch.equal(ops.embed(table, ids, prev, torch.zeros(1, dtype=torch.int32)),
                       table[[1, 2, 3]])
    assert torch.equal(ops.embed(table, ids, prev, torch.ones(1, dtype=torch.int32)),
                       table[[7, 8, 9]])


def test_build_is_content_hashed(tmp_path, monkeypatch):
    """Staleness is decided by source CONTENT: the built library embeds the hash of the
    sources it came from, and any source edit changes the hash the loader expects."""
    import shutil

    from agentic_traffic_testing_amd import ops

    build.build_kernels()
    assert ops.library_build_hash() == build.kernel_source_hash()
    copy = tmp_path / "csrc"
    shutil.copytree(build.CSRC, copy)
    before = build.kernel_source_hash()
    monkeypatch.setattr(build, "CSRC", copy)
    assert build.kernel_source_hash() == before  # same bytes, other place/mtime
    (copy / "common.h").write_text((copy / "common.h").read_text() + "\n// edit\n")
    assert build.kernel_source_hash() != before


def test_runtime_embeds_source_hash():
    from agentic_traffic_testing_amd import runtime

    assert runtime.BUILD_HASH == build.runtime_source_hash()


def test_current_library_is_used_without_object_files(tmp_path, monkeypatch):
    """A gpurun snapshot ships the .so but not _build/*.o: a library that embeds the current
    source hash must load as is (no rebuild - N DP ranks import at once), and a stale one is
    detected from its bytes."""
    from agentic_traffic_testing_amd import ops

    build.build_kernels()
    assert ops._lib_embeds(build.kernel_source_hash())
    assert not ops._lib_embeds("0" * 32)
    calls = []
    monkeypatch.setattr(build, "build_kernels", lambda *a, **k: calls.append(1))
    monkeypatch.setattr(ops, "_loaded", False)
    assert ops.load_native(build_if_missing=True), ops._load_error
    assert calls == []


def test_build_lock_serialises_processes(tmp_path):
    """Two processes holding the build lock never overlap."""
    import subprocess
    import sys

    log = tmp_path / "log"
    code = (
        "import time, sys\n"
        "from agentic_traffic_testing_amd.ops import build\n"
        "with build._build_lock():\n"
        f"    open({str(log)!r}, 'a').write('in\\n'); time.sleep(0.5)\n"
        f"    open({str(log)!r}, 'a').write('out\\n')\n")
    ps = [subprocess.Popen([sys.executable, "-c", code]) for _ in range(2)]
    assert all(p.wait(timeout=60) == 0 for p in ps)
    assert log.read_text().split() == ["in", "out", "in", "out"]


def test_hip_units_are_compiled_without_packed_fp32(tmp_path, monkeypatch):
    """Every HIP translation unit of both libraries: some packed fp32 instruction forms have given wrong results."""
    commands = []

    def run(cmd):
        commands.append(cmd)
        return types.SimpleNamespace(stdout="", stderr="", returncode=0)

    monkeypatch.setattr(build, "_run", run)
    monkeypatch.setattr(build, "BUILD", tmp_path)
    monkeypatch.setattr(build, "KERNEL_SO", tmp_path / "kernels.so")
    monkeypatch.setattr(build, "MIXER_SO", tmp_path / "mixers.so")
    build._build_kernels(True, 1, False)
    build._build_mixers(True, 1, False)
    units = [c for c in commands if any(str(x).endswith(".hip") for x in c)]
    assert len(units) == sum(len(list(d.glob("*.hip"))) for d in (build.CSRC, build.MIX_CSRC))
    for c in units:
        at = c.index("-packed-fp32-ops")
        assert c[at - 3:at] == ["-Xclang", "-target-feature", "-Xclang"]


def test_transfers_to_lds_read_their_base_behind_a_scalar_move():
    """A memory instruction in assembly that takes its address from a scalar register: the compiler does not keep the five
    wait states behind a vector instruction that wrote it (a reload of a spilled register), so the assembly moves it first."""
    found = 0
    for src in [*build.kernel_sources(), *build.mixer_sources()]:
        for text in re.findall(r'asm volatile\("((?:[^"\\]|\\.)*)"', src.read_text()):
            lines = text.split("\\n\\t")
            for i, line in enumerate(lines):
                if re.match(r"(global|buffer|scratch)_", line):
                    found += 1
                    base = line.split()[-1]
                    assert any(re.match(rf"s_mov_b64 {base},", x) for x in lines[:i]), (src.name, text)
    assert found == 3


def test_flash_kernels_share_their_assembly():
    """The two flash kernels are in libraries of their own and have the same assembly: what is mended in one is in the other."""
    def texts(name):
        src = next(p for p in [*build.kernel_sources(), *build.mixer_sources()] if p.name == name).read_text()
        return set(re.findall(r'asm volatile\(("(?:[^"\\]|\\.)*"(?:\s*"(?:[^"\\]|\\.)*")*)', src))

    llama, mixers = texts("flash_prefill.hip"), texts("sink_flash.hip")
    assert len(llama) >= 3
    # (4-byte transfers are the mixers' alone)
    assert mixers - llama == {t for t in mixers if "global_load_lds_dword %1" in t} and llama <= mixers


def code_objects(so):
    """The gfx950 code objects of a library built here."""
    data = Path(so).read_bytes()
    for start in (m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)):
        at = start + 32
        for _ in range(struct.unpack_from("<Q", data, start + 24)[0]):
            offset, size, n = struct.unpack_from("<3Q", data, at)
            if b"gfx950" in data[at + 24:at + 24 + n]:
                yield data[start + offset:start + offset + size]
            at += 24 + n


def llvm(tool, *args):
    path = Path(build.ROCM) / "llvm/bin" / tool
    if not path.exists():
        pytest.skip(f"no {tool}")
    return subprocess.run([path, *args], capture_output=True, text=True, check=True).stdout


def kernel_resources(so, tmp_path):
    """{kernel: its metadata's numbers} of a library built here."""
    found = {}
    for code in code_objects(so):
        (tmp_path / "object").write_bytes(code)
        for kernel in llvm("llvm-readelf", "--notes", tmp_path / "object").split("- .agpr_count:")[1:]:
            values = dict(re.findall(r"\.(\w+): +(\S+)", kernel))
            found[values["name"]] = {k: int(v) for k, v in values.items() if v.isdigit()}
    return found


def test_walk_of_the_recurrences_keeps_to_its_registers(tmp_path):
    """Without a delta rule nothing of the walk's is in scratch where a workgroup has a CU to itself, keys of 65 - 128 channels;
    narrower ones, one tile of columns per wave: two workgroups of eight waves fit on a CU, by registers and LDS."""
    wide = narrow = 0
    for name, r in kernel_resources(build.build_mixers(), tmp_path).items():
        m = re.search(r"scan_(?:walk|segments|segments_end)_kernelI(?:f|DF16b)Li(\d)ELi(\d+)ELi\dELi(\d)E", name)
        if m is None:
            continue
        mode, keys, tiles = map(int, m.groups())
        if mode < 3 and keys == 128:
            wide += 1
            assert r["private_segment_fixed_size"] == 0, (name, r)
        if keys == 64 and tiles == 1:
            narrow += 1
            assert r["vgpr_count"] <= 512 // 4 and 2 * r["group_segment_fixed_size"] <= 160 * 1024, (name, r)
    # (forms, types, alignments, tiles, kernels)
    assert wide >= 3 * 2 * 3 * 2 * 3 and narrow >= 3 * 2 * 2 * 3 + 2 * 2


def products_added_at_once(lines):
    """Matrix products of 32 terms that add to the result of one of 16 which no vector instruction has used in between."""
    def registers(x):
        m = re.match(r"v\[(\d+):(\d+)\]$", x) or re.match(r"v((\d+))$", x)
        return range(int(m[1]), int(m[2]) + 1) if m else ()

    fresh = set()
    for line in lines:
        op, _, args = line.split("//")[0].strip().partition(" ")
        if not op.startswith("v_"):
            if line.endswith(">:"):
                fresh.clear()
            continue
        if not fresh and not op.startswith("v_mfma_f32_16x16x16"):
            continue
        args = [x.strip() for x in args.split(",")]
        if op.startswith("v_mfma_f32_16x16x16"):
            fresh.update(registers(args[0]))
        elif op.startswith("v_mfma"):
            if "16x16x32" in op and fresh.intersection(registers(args[3])):
                yield line
            fresh.difference_update(registers(args[0]))
        else:
            for x in args:
                fresh.difference_update(registers(x))


def test_products_of_32_terms_wait_for_those_of_16(tmp_path):
    """The compiler leaves too few cycles between the two where nothing else reads the sum: the recurrences' kernels keep a
    vector instruction in between."""
    first, then = "v_mfma_f32_16x16x16_bf16 v[0:3], v[8:9], v[10:11], 0", "v_mfma_f32_16x16x32_bf16 v[4:7], v[12:15], v[16:19], v[0:3]"
    assert list(products_added_at_once([first, "s_nop 1", then])) == [then]
    assert not list(products_added_at_once([first, "v_fma_f32 v0, v0, v20, v21", "v_add_f32_e32 v30, v1, v2", "v_mov_b32_e32 v3, v3", then]))
    lines = pairs = 0
    for code in code_objects(build.build_mixers()):
        if b"scan_walk_kernel" in code:
            (tmp_path / "object").write_bytes(code)
            text = llvm("llvm-objdump", "-d", "--mcpu=gfx950", "--no-show-raw-insn", tmp_path / "object")
            lines += text.count("v_mfma_f32_16x16x16")
            pairs += len(list(products_added_at_once(text.split("\n"))))
    assert lines > 1000 and pairs == 0
