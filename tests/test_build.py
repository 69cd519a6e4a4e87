"""The kernel library's bookkeeping (no GPU, no compiler): which sources it belongs to and where it may go."""
import os
import re

from llm_infrence_engine_amd.kernels import build


def test_source_hash_names_the_sources_and_the_flags(monkeypatch):
    h = build.source_hash()
    assert re.fullmatch(r"[0-9a-f]{12}", h) and h == build.source_hash()
    monkeypatch.setattr(build, "FLAGS", build.FLAGS + ["-DOTHER"])
    assert build.source_hash() != h


def test_fallback_folder_is_per_user_and_per_sources():
    d = build._fallback_dir()
    assert str(os.getuid()) in d.name and build.source_hash() in d.name


def test_stamp_lies_beside_the_library(tmp_path):
    assert build._stamp_of(tmp_path / build.LIB_NAME) == tmp_path / "libminiserve_gfx950.stamp"


def test_no_kernel_spills_registers_to_memory():
    """The compiler's own report for every kernel of the library: none keeps registers in scratch memory (a spill
    in a decode kernel has doubled its time before it was seen) and none asks for more static LDS than a block
    may have.  Compiles the device code of all sources (about 20 s); skipped where there is no hipcc."""
    import pytest

    try:
        build._hipcc()
    except build.KernelLibraryError:
        pytest.skip("no hipcc here")
    usage = build.resource_usage()
    assert len(usage) > 100
    spills = {k: v["scratch"] for k, v in usage.items() if v.get("scratch", 0) > 0}
    assert not spills, f"kernels that spill registers: {spills}"
    assert all(v.get("lds", 0) <= 64 * 1024 for v in usage.values())
    # launches of more blocks than CUs, of four waves each, that count on a CU holding two of them
    pairs = {k: v["occupancy"] for k, v in usage.items() if re.search(r"attention_mfma_kernelILi128ELi1ELi4ELb0ELi1ELb[01]ELi0ELb0E", k)}
    assert len(pairs) == 2 and min(pairs.values()) >= 2, pairs


def test_a_written_barrier_waits_for_the_reads_before_it():
    """A barrier written in assembly, unlike ``__syncthreads``, waits for nothing by itself.  Behind it other waves load into
    the part of LDS that was read before it, so it has to name the reads (lgkmcnt) beside the loads (vmcnt): the products that
    use what was read, and the compiler's wait with them, may stand on either side of it."""
    found = []
    for src in build.sources():
        found += [(src.name, text) for text in re.findall(r'asm volatile\("([^"]*)"', src.read_text()) if "s_barrier" in text]
    assert found
    for name, text in found:
        assert re.search(r"s_waitcnt vmcnt\([^)]*\) lgkmcnt\(0\)\\n\\ts_barrier", text), (name, text)


def test_a_library_older_than_its_sources_is_built_again_not_loaded(tmp_path, monkeypatch):
    """``load()`` with a stamp that names other sources calls ``build()`` and loads what that returns."""
    import ctypes

    old = tmp_path / build.LIB_NAME
    old.write_bytes(b"not a library")
    build._stamp_of(old).write_text("0123456789ab\n")
    fresh = tmp_path / "fresh" / build.LIB_NAME
    calls, loaded = [], []

    def fake_build(verbose=True):
        calls.append(1)
        return fresh

    monkeypatch.setattr(build, "_lib", None)
    monkeypatch.setattr(build, "library_path", lambda: old)
    monkeypatch.setattr(build, "build", fake_build)
    monkeypatch.setattr(ctypes, "CDLL", lambda p: loaded.append(p) or object())
    build.load()
    assert calls == [1] and loaded == [str(fresh)]
    # a stamp that names these sources: loaded as it is
    build._stamp_of(old).write_text(build.source_hash() + "\n")
    monkeypatch.setattr(build, "_lib", None)
    build.load()
    assert calls == [1] and loaded[-1] == str(old)
    monkeypatch.setattr(build, "_lib", None)


def test_loads_written_in_assembly_wait_for_their_bases():
    """A memory instruction may read a scalar register five wait states after a vector instruction (the compiler's v_readlane)
    wrote it, which the compiler does not see to for assembly; and a load's registers are taken as written where its block
    ends.  So a block with loads begins with the wait states and ends with the wait for the loads."""
    for src in build.sources():
        text = src.read_text()
        for name, body in re.findall(r'#define (\w+)[^\n]*?("[^"\n]*(?:global|buffer|flat)_load[^\n]*)', text):
            blocks = [b for b in re.findall(r"asm volatile\((.*?)\s*:", text, re.S) if re.search(rf"\b{name}\(", b)]
            assert blocks, (src.name, name)
            for b in blocks:
                assert b.startswith("SGPRS_READY") and b.endswith('"s_waitcnt vmcnt(0)"'), (src.name, b)
            assert '#define SGPRS_READY "s_nop 4' in text
        assert not re.search(r'asm volatile\(\s*"[^"]*_(load|store)', text), src.name     # none beside those


def test_waits_of_one_item_keep_their_verdicts_apart():
    """A wave reads the verdict of a wait behind the wait's barrier, and nothing holds it up against the next wait's store: so
    the waits of one item of a decode chain have a word each, and none the one for waits that are the waves' own."""
    text = next(s for s in build.sources() if s.name == "decode_chain.hip").read_text()
    items = re.split(r"\n__device__ __forceinline__ bool run_", text)[1:]
    verdicts = [[int(v or 0) for v in re.findall(r"wait_first(?:<(\d+)>)?\(", i)] for i in items]
    assert sum(map(len, verdicts)) >= 6
    for v in verdicts:
        assert len(set(v)) == len(v) and 1 not in v
    assert f"int late[{max(map(max, filter(None, verdicts))) + 1}];" in text
