"""Host-side checks that need no GPU: the C-ABI library loads, exports every symbol the header
declares, and rejects bad shapes/handles before touching a device."""
import ctypes as C
import os
import re

import pytest

from openagents_amd import _ffi, backend

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    return _ffi.load()


def header_functions():
    text = open(os.path.join(ROOT, "include", "psn.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(psn_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol(lib):
    names = header_functions()
    assert len(names) >= 30
    for n in names:
        assert hasattr(lib, n), f"{n} declared in include/psn.h but not exported"
        assert n in _ffi.SIGNATURES, f"{n} has no ctypes signature"
    assert sorted(_ffi.SIGNATURES) == names
    assert lib.psn_abi_version() == 1


def test_block_geometry(lib):
    assert [lib.psn_block_bytes(t) for t in (_ffi.Q8_0, _ffi.Q4_0, _ffi.Q4_K, _ffi.Q6_K, _ffi.Q8_K)] == [34, 18, 144, 210, 292]
    assert [lib.psn_block_elems(t) for t in (_ffi.Q8_0, _ffi.Q4_0, _ffi.Q4_K, _ffi.Q6_K)] == [32, 32, 256, 256]
    assert backend.row_bytes(_ffi.Q4_0, 4096) == 2304
    assert backend.row_bytes(_ffi.Q4_K, 14336) == 8064
    assert backend.row_bytes(_ffi.Q6_K, 4096) == 3360
    with pytest.raises(backend.PsnError) as e:
        backend.row_bytes(_ffi.Q4_K, 4096 + 32)
    assert e.value.code == _ffi.E_SHAPE and "multiple" in str(e.value)
    with pytest.raises(backend.PsnError) as e:
        backend.row_bytes(99, 4096)
    assert e.value.code == _ffi.E_UNSUPPORTED


def test_activation_layout(lib):
    li = backend.actq_layout(_ffi.Q8_0, 4096, 1)
    assert (li.off_qs, li.off_d, li.off_s) == (0, 4096, 4096 + 512) and li.bytes == 4096 + 512 + 512
    li = backend.actq_layout(_ffi.Q8_K, 14336, 8)
    assert li.off_d == 8 * 14336 and li.off_d % 256 == 0 and li.off_s % 256 == 0
    assert li.bytes >= li.off_s + 8 * (14336 // 16) * 2
    assert backend.act_type_for(_ffi.Q4_0) == _ffi.Q8_0 and backend.act_type_for(_ffi.Q6_K) == _ffi.Q8_K
    for bad in (0, 9):
        with pytest.raises(backend.PsnError) as e:
            backend.actq_layout(_ffi.Q8_0, 4096, bad)
        assert e.value.code == _ffi.E_SHAPE
    with pytest.raises(backend.PsnError) as e:
        backend.actq_layout(_ffi.Q4_0, 4096, 1)
    assert e.value.code == _ffi.E_UNSUPPORTED


def test_matvec_plan_is_host_arithmetic(lib):
    for qt in (_ffi.Q4_0, _ffi.Q8_0, _ffi.Q4_K, _ffi.Q5_K, _ffi.Q6_K):
        for (n, k) in ((4096, 4096), (1024, 4096), (14336, 4096), (4096, 14336), (128256, 4096), (1, 256)):
            for batch in range(1, 9):
                for scheme in (_ffi.ACT_F32, _ffi.ACT_Q8):
                    p = backend.matvec_plan(qt, scheme, n, k, batch)
                    assert p.lanes_per_row in (8, 16, 32, 64) and p.rows_in_flight == 1
                    assert p.batch_tile >= batch and p.batch_tile in (1, 2, 4, 8)
                    assert 1 <= p.blocks <= 256 * 16
                    assert p.threads in (256, 512) or (p.stream and not p.mfma and p.threads in (320, 384, 448))
                    assert p.mfma in (0, 1, 2, 4, 8) and (p.mfma == 0 or (batch >= 2 and scheme == _ffi.ACT_Q8 and qt in (_ffi.Q4_K, _ffi.Q5_K)))
    for args, code in (((_ffi.Q4_0, 1, 0, 4096, 1), _ffi.E_SHAPE), ((_ffi.Q4_0, 1, 16, 4096 + 32, 1), _ffi.E_SHAPE),
                       ((_ffi.Q4_0, 1, 16, 4096, 9), _ffi.E_SHAPE), ((_ffi.Q8_K, 1, 16, 4096, 1), _ffi.E_UNSUPPORTED),
                       ((_ffi.Q4_0, 5, 16, 4096, 1), _ffi.E_UNSUPPORTED)):
        with pytest.raises(backend.PsnError) as e:
            backend.matvec_plan(*args)
        assert e.value.code == code, args


def test_matvec_plans_are_consistent_over_many_shapes(lib):
    """Host arithmetic only: every plan the library returns over a grid of shapes and batches is one its own
    kernels accept (thread counts, slice arithmetic of the MFMA kernels, enough workgroups for one-unit waves)."""
    for qt in (_ffi.Q4_0, _ffi.Q8_0, _ffi.Q4_K, _ffi.Q5_K, _ffi.Q6_K):
        for k in (256, 512, 768, 1024, 2048, 2304, 4096, 5120, 8192, 11008, 14336, 16384, 28672):
            for n in (1, 16, 17, 48, 1000, 1024, 4096, 14336, 128256):
                for batch in (1, 2, 3, 5, 8):
                    for x_is_f32 in (False, True):
                        p = backend.matvec_plan(qt, _ffi.ACT_Q8, n, k, batch, 256, x_is_f32)
                        assert 1 <= p.blocks <= 1 << 20, p.as_dict()
                        # four or eight waves; the batch-1 streaming kernels also take five to seven
                        assert p.threads in (256, 512) or (p.stream and not p.mfma and p.threads in (320, 384, 448)), p.as_dict()
                        if p.mfma:
                            c, waves = k // 256, p.threads // 64
                            assert qt in (_ffi.Q4_K, _ffi.Q5_K) and batch >= 2 and n % 16 == 0, p.as_dict()
                            assert p.mfma in (1, 2, 4, 8) and p.mfma <= waves and c % p.mfma == 0 and c // p.mfma <= 8, p.as_dict()
                            assert p.stage_lds == 1 and p.stream == 1, p.as_dict()
                            if c // p.mfma > 4:
                                assert p.blocks * (waves // p.mfma) >= n // 16, p.as_dict()      # one wave per unit
                            lds = c * 160 + waves * 1024 + waves * (9 if qt == _ffi.Q4_K else 11) * 1024
                            assert lds <= 160 * 1024, p.as_dict()
                        elif p.stream:
                            assert batch == 1 and p.stage_lds in (1, 2) and k // 256 <= p.lanes_per_row, p.as_dict()
                            npass = n // (64 // p.lanes_per_row)
                            if 4 * 256 < npass <= 8 * 256 and p.threads < 512:
                                # one pass per wave, one workgroup on every compute unit
                                assert p.blocks == 256 and p.blocks * (p.threads // 64) >= npass, p.as_dict()
    # Llama-3-8B's fused q/k/v projection: 6144 rows of sixteen chunks, four rows a pass -> 1536 passes = 256 x 6 waves
    p = backend.matvec_plan(_ffi.Q4_0, _ffi.ACT_Q8, 6144, 4096, 1, 256, True)
    assert (p.stream > 0, p.threads, p.blocks) == (True, 384, 256), p.as_dict()


def test_swiglu_fused_launch_check_is_host_arithmetic(lib):
    """psn_qmatvec_norm_swiglu_check: which gate|up shapes the SwiGLU-fused launch serves, without a device."""
    chk = lambda qt, n, k: int(lib.psn_qmatvec_norm_swiglu_check(qt, n, k, 256))
    for qt in (_ffi.Q4_0, _ffi.Q8_0, _ffi.Q4_K, _ffi.Q5_K, _ffi.Q6_K):
        assert chk(qt, 14336, 4096) == 0 and chk(qt, 1024, 2048) == 0
        assert chk(qt, 4096, 14336) == _ffi.E_UNSUPPORTED              # rows longer than the fused staging holds
        assert chk(qt, 1026, 4096) == _ffi.E_UNSUPPORTED               # not whole passes
        assert chk(qt, 0, 4096) == _ffi.E_SHAPE and chk(qt, 1024, 4100) == _ffi.E_SHAPE
    assert chk(_ffi.Q6_K, 1024, 2304) == _ffi.E_UNSUPPORTED            # 210-byte blocks: rows of whole 16-byte words only
    assert chk(_ffi.Q8_K, 1024, 4096) != 0                             # not a weight format


def test_prefill_plans_are_consistent_over_many_shapes(lib):
    """Host arithmetic only: every prefill plan over a grid of shapes is one psn_qmatmul_prefill_tiled accepts --
    a known tile, a family the format has, a K split that leaves whole chunks per range and an atomically addable Y."""
    tiles = {(64, 64), (64, 128), (128, 128), (128, 256), (256, 128), (256, 256)}
    for qt in (_ffi.Q4_0, _ffi.Q8_0, _ffi.Q4_K, _ffi.Q5_K, _ffi.Q6_K):
        for k in (256, 512, 1024, 2048, 2304, 4096, 5120, 8192, 11008, 14336):
            for n in (1, 17, 64, 130, 1000, 1024, 4096, 6144, 14336):
                for m in (1, 7, 64, 65, 128, 200, 512, 777, 2048, 4096):
                    tm, tn, sp, wv = backend.prefill_plan(m, n, k, 256, qt)
                    tag = (qt, m, n, k, tm, tn, sp, wv)
                    assert (tm, tn) in tiles and sp in (1, 2, 4, 8), tag
                    if sp > 1:
                        assert (m * n) % 4 == 0 and k // 256 >= 2 * sp, tag
                    if m <= 64 and (qt != _ffi.Q6_K or k % 2048 == 0):
                        assert wv == 64 and (tm, tn) == (64, 64), tag           # the weight-streaming kernel
                    else:
                        assert wv != 64, tag
                    if wv == 128:
                        assert m > 64 and tn == 256 and tm in (128, 256) and sp <= 4, tag
                    elif wv == 32:
                        assert qt in (_ffi.Q4_0, _ffi.Q8_0) and (tm, tn) == (256, 256), tag
                    elif wv == 16:
                        assert (tm, tn) in {(64, 64), (64, 128), (128, 128), (128, 256)}, tag
                        assert qt in (_ffi.Q4_0, _ffi.Q8_0) or (qt != _ffi.Q6_K and (tm, tn) == (128, 256)), tag
                    else:
                        assert wv in (4, 64), tag


def test_plans_for_at_most_64_rows_cut_k_for_the_kernel_they_name(lib):
    """The plan for M <= 64 names the 64 x 64 kernel: its K split is the one that kernel needs, doubled only while the workgroups leave half
    of the compute units idle, whatever psn_qmatmul_prefill runs there itself."""
    for qt in (_ffi.Q4_0, _ffi.Q8_0, _ffi.Q4_K, _ffi.Q5_K, _ffi.Q6_K):
        for n, k in ((1024, 4096), (4096, 4096), (4096, 14336), (14336, 4096), (1000, 2048), (17, 8192), (300, 2304)):
            if qt == _ffi.Q6_K and k % 2048:
                continue
            for m in (1, 16, 33, 48, 64):
                want = 1
                while want < 8 and -(-n // 64) * want * 2 <= 256 and k // 256 >= 4 * want and (m * n) % 4 == 0:
                    want *= 2
                assert backend.prefill_plan(m, n, k, 256, qt) == (64, 64, want, 64), (qt, m, n, k)


def test_prefill_choice_is_the_plan_or_a_thin_kernel(lib):
    """Host arithmetic: for more than 64 rows the choice is the plan; for fewer it is that or a thin kernel that exists, tall enough for X, with
    a K split that leaves two whole chunks per range; without a workspace it is never the dense family."""
    thin = 0
    for qt in (_ffi.Q4_0, _ffi.Q8_0, _ffi.Q4_K, _ffi.Q5_K, _ffi.Q6_K):
        for k in (256, 768, 2048, 4096, 11008, 14336):
            for n in (1, 17, 1000, 1024, 4096, 14336):
                for m in (1, 16, 17, 33, 64, 65, 512, 4096):
                    tm, tn, sp, wv = c = backend.prefill_choice(m, n, k, qt)
                    if wv == 8:
                        thin += 1
                        assert m <= tm <= 64 and tm - m < 16 and tn in (16, 32, 64), (qt, m, n, k, c)
                        assert tn < 64 or tm in {_ffi.Q8_0: (16,), _ffi.Q6_K: (16, 32, 48)}.get(qt, (32, 48)), (qt, m, n, k, c)
                        assert sp == 1 or ((m * n) % 4 == 0 and k // 256 >= 2 * sp), (qt, m, n, k, c)
                    else:
                        assert c == backend.prefill_plan(m, n, k, 256, qt), (qt, m, n, k, c)
                    assert backend.prefill_choice(m, n, k, qt, workspace=False)[3] != 128
    assert thin
    assert lib.psn_qmatmul_prefill_choice(_ffi.Q4_0, 1, 1, 100, 256, 1, *[C.byref(C.c_int32()) for _ in range(4)]) == _ffi.E_SHAPE
    assert lib.psn_qmatmul_prefill_choice(_ffi.Q4_0, 1, 1, 256, 256, 1, None, None, None, None) == _ffi.E_INVALID_ARG


def test_few_rows_over_wide_matrices_take_a_kernel_that_exists(lib):
    """Host arithmetic, more weight rows than 64 per compute unit: the choice for M <= 64 is the 64 x 64 kernel, a thin one, or an eight-wave tile of family 4, with a K split
    that leaves two whole chunks per range, and family 4 is taken somewhere in every format; up to 64 rows per unit it is not (Q6_K rows of odd sizes aside)."""
    for qt in (_ffi.Q4_0, _ffi.Q8_0, _ffi.Q4_K, _ffi.Q5_K, _ffi.Q6_K):
        families = set()
        for k in (256, 768, 2048, 5120, 8192):
            for n in (16384, 16385, 18176, 28672, 128256):
                for m in (1, 16, 17, 33, 48, 64):
                    tm, tn, sp, wv = c = backend.prefill_choice(m, n, k, qt)
                    assert wv in (4, 8, 64) and sp in (1, 2, 4, 8), (qt, m, n, k, c)
                    assert wv != 4 or ((tm, tn) in {(64, 64), (64, 128), (128, 128), (256, 128)} and (n > 16384 or (qt == _ffi.Q6_K and k % 2048))), (qt, m, n, k, c)
                    assert wv != 64 or (c[:2] == (64, 64) and (qt != _ffi.Q6_K or k % 2048 == 0)), (qt, m, n, k, c)
                    assert sp == 1 or ((m * n) % 4 == 0 and k // 256 >= 2 * sp), (qt, m, n, k, c)
                    families.add(wv)
        assert 4 in families and 8 in families, (qt, families)


def test_null_handles_are_rejected_without_a_device(lib):
    assert lib.psn_stream_sync(None) == _ffi.E_INVALID_ARG
    assert lib.psn_buf_free(None) == _ffi.E_INVALID_ARG
    assert lib.psn_module_unload(None) == _ffi.E_INVALID_ARG
    assert lib.psn_ctx_destroy(None) == _ffi.E_INVALID_ARG
    assert lib.psn_qmatvec(None, None, _ffi.Q4_0, 0, 1, None, None, None, 16, 4096, 1) == _ffi.E_INVALID_ARG
    assert b"null" in lib.psn_last_error()
    assert lib.psn_qmatvec(None, None, _ffi.Q4_0, 7, 1, None, None, None, 16, 4096, 1) == _ffi.E_UNSUPPORTED
    h = C.c_void_p()
    assert lib.psn_buf_alloc(None, 16, C.byref(h)) == _ffi.E_INVALID_ARG and not h.value
    assert lib.psn_module_load(None, None, 0, C.byref(h)) == _ffi.E_INVALID_ARG
    assert lib.psn_error_name(-4) == b"PSN_E_NO_DEVICE"


def test_context_creation_fails_loudly_without_gfx950(lib):
    h = C.c_void_p()
    rc = lib.psn_ctx_create(0, C.byref(h))
    if rc == 0:                      # running on a GPU box: nothing to assert about absence
        assert lib.psn_ctx_destroy(h) == 0
        return
    assert rc == _ffi.E_NO_DEVICE and not h.value
    assert lib.psn_last_error()
    with pytest.raises(backend.PsnError):
        backend.HipBackend(0)


def test_missing_library_is_an_error_not_a_fallback(monkeypatch):
    monkeypatch.setattr(_ffi, "_lib", None)
    monkeypatch.setattr(_ffi, "LIB_PATH", "/nonexistent/libpsn_hip.so")
    with pytest.raises(_ffi.LibraryMissing):
        _ffi.load()


def test_integration_doc_binding_lists_every_entry_point():
    """The Rust `-sys` text a maintainer would paste must not drift from the header."""
    doc = open(os.path.join(ROOT, "INTEGRATION.md")).read()
    rust = set(re.findall(r"pub fn (psn_[a-z0-9_]+)\(", doc))
    assert rust == set(header_functions())


def test_static_scratch_is_exported_by_the_device_image():
    """The no-allocation entry point finds its scratch with hipGetSymbolAddress, which looks the
    registered name up among the symbols the gfx950 image EXPORTS; a file-local symbol there makes the
    runtime abort.  Checked on the built object, no GPU needed."""
    import shutil
    import subprocess
    import tempfile
    obj = os.path.join(ROOT, "openagents_amd", "lib", "psn_noalloc.o")
    bundler, readelf = "/opt/rocm/llvm/bin/clang-offload-bundler", "/opt/rocm/llvm/bin/llvm-readelf"
    if not (os.path.exists(obj) and os.path.exists(bundler) and os.path.exists(readelf) and shutil.which("objcopy")):
        pytest.skip("built object or LLVM binutils not present")
    with tempfile.TemporaryDirectory() as d:
        fat, elf = os.path.join(d, "fat.bin"), os.path.join(d, "dev.elf")
        subprocess.check_call(["objcopy", "-O", "binary", "--only-section=.hip_fatbin", obj, fat])
        subprocess.check_call([bundler, "--unbundle", "--type=o", f"--input={fat}", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={elf}"])
        syms = subprocess.check_output([readelf, "--dyn-syms", elf], text=True)
    rows = [ln.split() for ln in syms.splitlines() if ln.strip().endswith("scratch")]
    assert rows, syms
    assert all(r[3] == "OBJECT" and r[4] == "GLOBAL" and int(r[2]) == 1 << 20 for r in rows), rows


def _kernel_notes():
    """(name, lookup of a field) for every kernel of every built code object, from the code objects' own metadata notes."""
    import glob
    import subprocess
    import tempfile
    bundler, readelf = "/opt/rocm/llvm/bin/clang-offload-bundler", "/opt/rocm/llvm/bin/llvm-readelf"
    objs = sorted(glob.glob(os.path.join(ROOT, "openagents_amd", "lib", "*.gfx950.hsaco")))
    if not objs or not (os.path.exists(bundler) and os.path.exists(readelf)):
        pytest.skip("built code objects or LLVM binutils not present")
    out = []
    with tempfile.TemporaryDirectory() as d:
        for path in objs:
            elf = os.path.join(d, os.path.basename(path) + ".elf")
            subprocess.check_call([bundler, "--unbundle", "--type=o", f"--input={path}", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={elf}"])
            notes = subprocess.check_output([readelf, "--notes", elf], text=True)
            for blk in notes.split("- .agpr_count:")[1:]:
                get = lambda key, blk=blk: re.search(r"\." + key + r":\s+(\S+)", blk).group(1)
                out.append((get("name"), get))
    return out


def _kernel_resources():
    """name -> (vgpr spills, sgpr spills, scratch bytes per lane)"""
    return {name: (int(get("vgpr_spill_count")), int(get("sgpr_spill_count")), int(get("private_segment_fixed_size"))) for name, get in _kernel_notes()}


def _kernel_registers():
    return {name: int(get("vgpr_count")) for name, get in _kernel_notes()}


def test_no_kernel_spills_registers_or_uses_scratch():
    """Every kernel a planner can return (and every other kernel of the library) keeps its working set in
    registers: a spilled register or a scratch copy of the kernel arguments costs memory round trips in the
    middle of a stream and has gone unnoticed before."""
    res = _kernel_resources()
    assert len(res) > 300
    for family in ("psn_mvs_q4_0_q8_g16_xf_s2", "psn_mvs_q6_K_q8_g16_lds_s1", "psn_prefill_q4_0_skinny", "psn_prefill_q8_0_m128_n256_ws",
                   "psn_prefill_q4_0_m256_n256", "psn_attn_partial_rope", "psn_mv_q4_K_q8_g16_r1_b8_lds"):
        assert family in res, family
    bad = {k: v for k, v in res.items() if v != (0, 0, 0)}
    assert not bad, bad


def _prefill_lds(calls):
    """what expressions of psn_prefill_lds.h come to: the sizes that the host launches with and that the kernels assert their layouts to equal"""
    import subprocess
    import tempfile
    with tempfile.TemporaryDirectory() as d:
        src = os.path.join(d, "lds.cpp")
        with open(src, "w") as f:
            f.write('#include "psn_prefill_lds.h"\n#include <cstdio>\nint main() {\n' + "".join(f'    std::printf("%d\\n", (int)({c}));\n' for c in calls) + "}\n")
        subprocess.check_call(["g++", "-std=c++17", "-I", os.path.join(ROOT, "openagents_amd", "csrc"), "-o", os.path.join(d, "lds"), src])
        return [int(v) for v in subprocess.check_output([os.path.join(d, "lds")], text=True).split()]


def test_prefill_planner_counts_the_workgroups_a_compute_unit_can_hold():
    """The cost models' workgroups per compute unit against the built kernels: 512 vector registers per lane and SIMD, given out in eights, two waves of a workgroup on each of the four
    SIMDs, and 160 KB of LDS.  Family 4's table holds what the registers allow (the planner takes the LDS of the format beside it), the dense family's and the thin kernels' rule
    what both do."""
    src = open(os.path.join(ROOT, "openagents_amd", "csrc", "psn_host.cpp")).read()
    table = lambda name: re.search(name + r"\[\] = \{(.*?)\n\};", src, re.S).group(1)
    tiles = re.findall(r"\{(\d+), (\d+)\}", re.search(r"k_prefill_tiles\[\]\[2\] = \{(.*)\};", src).group(1))
    regs = _kernel_registers()
    by_registers = lambda name: 512 // (-(-regs[name] // 8) * 8) // 2
    formats = ("q4_0", "q8_0", "q4_K", "q5_K", "q6_K")
    in_loop = re.findall(r"\{(\d), (\d), (\d), \{", table("k_prefill_cost"))
    assert len(in_loop) == 4
    for tile, others, q6_K in in_loop:
        m, n = map(int, tiles[int(tile)])
        for fmt in formats:
            for kernel in ("_pp", "_pp32") if m == 256 else ("_pp",):
                assert by_registers(f"psn_prefill_{fmt}_m{m}_n{n}{kernel}") == int(q6_K if fmt == "q6_K" else others), (fmt, m, n)
    assert re.search(r"by_lds = PSN_LDS_MAX / psn_lds_in_loop\(format_index\(qtype\), bm, bn\);", src)

    dense = [tuple(map(int, t)) for name in ("k_dense_cost", "k_packed_cost") for t in re.findall(r"\{(\d+), (\d+), (\d), \{", table(name))]
    assert len(dense) == 7
    for (m, n, per_cu), lds in zip(dense, _prefill_lds(f"psn_lds_dense({m}, {n})" for m, n, _ in dense)):
        name = "psn_prefill_dense_f16" + ("" if m == 256 else "_m128" if n == 256 else f"_m{m}_n{n}")
        assert min(by_registers(name), 160 * 1024 // lds) == per_cu, (m, n)

    thin = [(name, *re.fullmatch(r"psn_prefill_(\w+)_thin_(\d)_(\d)", name).groups()) for name in regs if "_thin_" in name]
    assert len(thin) == 5 * 8 + 2 + 1 + 2 + 2 + 3
    for (name, fmt, tm, rt), lds in zip(thin, _prefill_lds(f"psn_lds_thin({formats.index(fmt)}, {tm}, {rt})" for _, fmt, tm, rt in thin)):
        two = tm == "1" and (rt == "1" or (rt == "2" and fmt not in ("q8_0", "q6_K")))
        assert min(by_registers(name), 160 * 1024 // lds) == (2 if two else 1), name


def test_prefill_lds_sizes_follow_from_the_layouts():
    """Restated from what lies in LDS: 64 x 128 tiles of family 4 are where a format decides whether two workgroups share a compute unit, and one thin kernel has no room for scales."""
    sizes = _prefill_lds([f"psn_lds_in_loop({f}, 64, 128)" for f in range(5)] + ["psn_lds_in_loop(2, 256, 128)", "psn_lds_thin(2, 3, 4)", "psn_lds_thin(3, 3, 4)", "psn_lds_thin_scales(3, 3, 4)",
                          "psn_lds_dense(64, 64)", "psn_lds_dense(256, 256)"])
    x = 2 * 64 * 256
    raw = lambda words, extra: 2 * ((128 * words // 64 + 1) * 1024 + extra)
    assert sizes[:5] == [x + raw(9, 0), x + raw(17, 0), x + raw(9, 0) + 8 * 1024, x + raw(11, 0) + 8 * 1024, x + raw(13, 128 * 8)]
    assert [160 * 1024 // v for v in sizes[:5]] == [2, 1, 2, 1, 1]
    assert sizes[5:] == [4 * 256 * 128 + 2 * 128 * 128, 8 * (64 * (144 + 64) + 3 * 2048), 8 * (64 * 176 + 3 * 2048), 0, 5 * 128 * 128, 160 * 1024]


def test_prefill_planner_knows_how_full_the_rounds_are(lib):
    """Shapes on which a planner that takes another deal of the tiles than the kernels', or is blind to how full a round is, picks the slower family (measured us, weights from
    memory): 5120 x 13824 M = 3072 dense 352 .. 367, in the loop 397 .. 453 (N tiles dealt to the XCDs in turn would make it two rounds); 32000 x 4096 M = 1024 in the loop 265,
    dense 284; 4096 x 4096 M = 4096 dense 115, in the loop 133; 1536 x 5632 M = 640 Q4_K 64 x 64 tiles 27.5, 128 x 128 41.  Without a workspace the dense family is out."""
    for qt in (_ffi.Q4_0, _ffi.Q8_0, _ffi.Q4_K, _ffi.Q5_K, _ffi.Q6_K):
        assert backend.prefill_choice(3072, 5120, 13824, qt) == (256, 256, 1, 128)
        assert backend.prefill_choice(3072, 5120, 13824, qt, workspace=False) == (256, 128, 1, 4)
    assert backend.prefill_choice(1024, 32000, 4096, _ffi.Q4_0) == (256, 128, 1, 4)
    assert backend.prefill_choice(4096, 4096, 4096, _ffi.Q4_0) == (256, 256, 1, 128)
    for qt in (_ffi.Q4_K, _ffi.Q5_K):
        assert backend.prefill_choice(640, 1536, 5632, qt)[:2] == (64, 64)


def test_prefill_planner_picks_a_plan_near_the_fastest_where_weights_come_from_memory(lib):
    """Measured us of the explicit plans (weight copies rotating through 320 MB, zero fill and dequantization pass included) for shapes that none of the cost models was fitted to
    and that a fit to weights out of the caches got wrong by 10 to 25 %, above all 64 x 64 tiles without a K cut: what is chosen is within 5 % of the fastest."""
    measured = {
        (_ffi.Q4_0, 117, 2816, 2816): {(64, 64, 2, 4): 11.9, (64, 128, 4, 4): 12.5, (64, 64, 4, 4): 12.7, (64, 64, 1, 4): 14.9},
        (_ffi.Q4_0, 227, 3968, 7936): {(64, 128, 2, 4): 31.0, (128, 128, 4, 4): 31.1, (64, 128, 4, 4): 32.7, (64, 64, 2, 4): 32.9, (64, 64, 1, 4): 38.6},
        (_ffi.Q6_K, 148, 2048, 2048): {(64, 64, 2, 4): 11.8, (64, 64, 4, 4): 12.8, (64, 128, 4, 4): 13.7, (64, 64, 1, 4): 13.9},
        (_ffi.Q4_K, 379, 1536, 4608): {(128, 128, 4, 4): 19.9, (64, 128, 2, 4): 20.5, (64, 64, 2, 4): 22.1, (64, 64, 1, 4): 22.9},
        (_ffi.Q5_K, 291, 1792, 4608): {(128, 128, 4, 4): 20.0, (64, 128, 2, 4): 22.0, (64, 64, 2, 4): 22.6, (64, 64, 1, 4): 23.1},
        (_ffi.Q8_0, 177, 2304, 2304): {(64, 64, 2, 4): 11.9, (64, 64, 1, 4): 13.6, (64, 64, 4, 4): 13.8, (64, 128, 4, 4): 14.5},
        (_ffi.Q6_K, 99, 4608, 4608): {(128, 128, 4, 4): 23.6, (64, 64, 2, 4): 25.9, (64, 64, 4, 4): 26.2, (64, 64, 1, 4): 26.7},
        (_ffi.Q4_0, 640, 1536, 5632): {(64, 128, 2, 4): 25.4, (64, 64, 2, 4): 25.5, (128, 128, 4, 4): 25.8, (64, 64, 1, 4): 28.0},
        (_ffi.Q4_K, 621, 7168, 18432): {(128, 128, 4, 4): 230.1, (128, 128, 2, 4): 233.2, (256, 128, 4, 4): 247.9, (256, 128, 1, 4): 263.2, (256, 256, 2, 128): 279.5},
        (_ffi.Q6_K, 2266, 7168, 24576): {(256, 256, 1, 128): 676.9, (256, 256, 2, 128): 744.1, (128, 256, 1, 128): 800.9, (256, 128, 1, 4): 820.1},
    }
    for (qt, m, n, k), us in measured.items():
        chosen = backend.prefill_choice(m, n, k, qt)
        assert us.get(chosen, 1e9) <= 1.05 * min(us.values()), (qt, m, n, k, chosen)


def test_packed_plans_name_a_tile_of_the_multiply_and_a_cut_that_may_be_made(lib):
    """Host arithmetic: every tile is taken somewhere, K is cut only where Y can be zeroed by 16-byte words and every range holds two chunks; what the call refuses, the plan refuses."""
    taken = set()
    for m in (1, 33, 64, 203, 512, 1281, 2048, 4001, 1 << 20):
        for n in (1, 66, 1000, 1024, 4097, 14336, 1 << 20):
            for k in (256, 1280, 4096, 14336):
                tm, tn, sp = backend.packed_plan(m, n, k)
                assert (tm, tn) in {(64, 64), (64, 128), (128, 128), (128, 256), (256, 256)}, (m, n, k)
                assert sp == 1 or (sp in (2, 4, 8) and (m * n) % 4 == 0 and k // 256 >= 2 * sp), (m, n, k, sp)
                taken.add((tm, tn))
    assert len(taken) == 5
    one = [C.c_int32() for _ in range(3)]
    assert lib.psn_qmatmul_prefill_packed_plan(1, 1, 300, 256, *map(C.byref, one)) == _ffi.E_SHAPE
    assert lib.psn_qmatmul_prefill_packed_plan(0, 1, 256, 256, *map(C.byref, one)) == _ffi.E_SHAPE
    assert lib.psn_qmatmul_prefill_packed_plan(1, 1, 256, 256, None, None, None) == _ffi.E_INVALID_ARG
    assert backend.packed_plan(512, 4096, 4096, 0) == backend.packed_plan(512, 4096, 4096, 256)


def test_prefill_plans_take_the_dense_family_only_for_large_m():
    """Host arithmetic: from a few thousand rows of X on every format is dequantized once and multiplied as
    fp16 (family 128, 256 x 256 or 128 x 256 tiles); 64 rows and fewer never are."""
    for qt in (_ffi.Q4_0, _ffi.Q8_0, _ffi.Q4_K, _ffi.Q5_K, _ffi.Q6_K):
        for n, k in ((14336, 4096), (4096, 14336)):
            tm, tn, sp, wv = backend.prefill_plan(4096, n, k, 256, qt)
            assert tm in (128, 256) and (tn, wv) == (256, 128) and sp in (1, 2, 4), (qt, n, k)
            for m in (1, 16, 64):
                assert backend.prefill_plan(m, n, k, 256, qt)[3] == 64     # 64 rows and fewer: the weight-streaming kernel
    assert backend.prefill_plan(64, 4096, 4096 + 256, 256, _ffi.Q6_K)[3] == 4   # Q6_K rows that are not whole 16-byte words
    lib = _ffi.load()
    assert lib.psn_error_name(lib.psn_prefill_reserve(None, 4096, 4096)) == b"PSN_E_INVALID_ARG"
