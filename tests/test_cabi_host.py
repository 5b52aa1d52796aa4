"""CPU-side checks of the C-ABI library: it loads, exports every symbol the
headers declare, and its host-only logic (cache bookkeeping, argument
validation) behaves like the reference.  No kernel is launched here."""

import ctypes as C
import os
import re

import pytest

from oracle import dflash_oracle as O
from swiftlm_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    names = set()
    for h in ("dflash_hip.h", "dflash_cache.h", "dflash_profile.h"):
        text = open(os.path.join(ROOT, "include", h)).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        names |= set(re.findall(r"\b(dflash_[a-z0-9_]+)\s*\(", text))
    return names


def test_library_exports_every_declared_symbol():
    lib = C.CDLL(_lib.LIB_PATH)
    declared = _declared_symbols()
    assert len(declared) >= 26
    for name in sorted(declared):
        assert hasattr(lib, name), f"{name} declared in include/ but not exported"
    assert declared == set(_lib.SIGNATURES), "ctypes table and headers disagree"


def test_version_and_error_text():
    lib = _lib.load()
    assert lib.dflash_version() == 100
    assert isinstance(_lib.last_error(), str)


def test_modulemap_names_the_header():
    mm = open(os.path.join(ROOT, "include", "module.modulemap")).read()
    assert 'header "dflash_hip.h"' in mm and 'header "dflash_cache.h"' in mm and 'link "dflash_hip"' in mm


# ---- cache bookkeeping (host only; device pointers are never dereferenced) ----


def _cache(kind):
    h = C.c_void_p(_lib.load().dflash_cache_create(kind, 4))
    assert h
    return h


def test_cache_create_rejects_bad_kind():
    assert not _lib.load().dflash_cache_create(9, 4)
    assert "bad kind" in _lib.last_error()


def test_cache_arm_snapshot_and_clear():
    lib = _lib.load()
    c = _cache(_lib.CACHE_TAPE)
    lib.dflash_cache_set_slot(c, 0, 0x1000)
    lib.dflash_cache_set_slot(c, 1, 0x2000)
    assert not lib.dflash_cache_is_armed(c)
    assert lib.dflash_cache_arm_rollback(c, 7) == 0
    assert lib.dflash_cache_is_armed(c)
    # rollback without a recorded tape restores the snapshot pointers and disarms
    lib.dflash_cache_set_slot(c, 0, 0x3000)
    lib.dflash_cache_set_slot(c, 1, 0x4000)
    assert lib.dflash_cache_rollback(c, None, 2) == 0
    assert lib.dflash_cache_get_slot(c, 0) == 0x1000 and lib.dflash_cache_get_slot(c, 1) == 0x2000
    assert not lib.dflash_cache_is_armed(c)
    # rollback when never armed is a no-op (RecurrentRollbackCache.swift:96-99)
    lib.dflash_cache_set_slot(c, 1, 0x5000)
    assert lib.dflash_cache_rollback(c, None, 0) == 0
    assert lib.dflash_cache_get_slot(c, 1) == 0x5000
    lib.dflash_cache_destroy(c)


def test_cache_rollback_requires_functional_update():
    lib = _lib.load()
    c = _cache(_lib.CACHE_TAPE)
    lib.dflash_cache_set_slot(c, 0, 0x1000)
    lib.dflash_cache_set_slot(c, 1, 0x2000)
    lib.dflash_cache_arm_rollback(c, 0)
    rc = lib.dflash_cache_record_tape(c, 0x10, _lib.F32, 0x20, 0x30, _lib.BF16, 3, None, 2, _lib.F32,
                                      1, 16, 16, 32, 128, 128, 0)
    assert rc == 0
    # slot 1 still points at the pre-verify buffer: refusing beats corrupting the snapshot
    assert lib.dflash_cache_rollback(c, None, 3) == _lib.INVALID
    assert "pre-verify" in _lib.last_error()
    # a refused rollback changes nothing: still armed, slots as they were, so the caller can correct and retry
    assert lib.dflash_cache_is_armed(c)
    assert lib.dflash_cache_get_slot(c, 0) == 0x1000 and lib.dflash_cache_get_slot(c, 1) == 0x2000
    lib.dflash_cache_destroy(c)


def test_refused_rollback_keeps_the_snapshots_tensors(monkeypatch):
    """A refused rollback leaves the handle armed and pointing at the snapshot, also where a slot holds another tensor by then: the
    cache object still holds the snapshot's until a rollback or clear_transients has let go of them."""
    from swiftlm_amd import RecurrentRollbackCache, rollback_cache

    monkeypatch.setattr(rollback_cache, "_stream", lambda: None)
    lib, c = _lib.load(), RecurrentRollbackCache()
    for slot, p in enumerate((0x1000, 0x2000)):
        lib.dflash_cache_set_slot(c._h, slot, p)
        c._by_ptr[p] = f"snapshot {slot}"
    c.arm_rollback(0)
    lib.dflash_cache_set_slot(c._h, 0, 0x3000)                 # a new window, but the state is still the pre-verify one
    c._by_ptr[0x3000] = "window"
    assert lib.dflash_cache_record_tape(c._h, 0x10, _lib.F32, 0x20, 0x30, _lib.BF16, 3, None, 2, _lib.F32, 1, 16, 16, 32, 128, 128, 0) == 0
    with pytest.raises(_lib.DFlashError, match="pre-verify"):
        c.rollback(3)
    assert c.is_armed and c._by_ptr == {0x1000: "snapshot 0", 0x2000: "snapshot 1", 0x3000: "window"}
    c.clear_transients()
    assert not c.is_armed and c._by_ptr == {0x2000: "snapshot 1", 0x3000: "window"}


def test_restore_validates_every_cache_before_touching_any():
    """A list whose LAST cache cannot be rolled back (slot 1 still holds the pre-verify buffer), or that holds a
    null handle, is refused as a whole: the caches before it keep their snapshot, tape, armed flag and offsets."""
    lib = _lib.load()
    good, kv, bad = _cache(_lib.CACHE_SNAPSHOT), _cache(_lib.CACHE_KV), _cache(_lib.CACHE_TAPE)
    lib.dflash_cache_set_slot(good, 1, 0x2000)
    lib.dflash_cache_arm_rollback(good, 100)
    lib.dflash_cache_set_slot(good, 1, 0x4000)
    lib.dflash_cache_set_offset(kv, 116)
    lib.dflash_cache_set_slot(bad, 0, 0x1000)
    lib.dflash_cache_set_slot(bad, 1, 0x2000)
    lib.dflash_cache_arm_rollback(bad, 100)
    assert lib.dflash_cache_record_tape(bad, 0x10, _lib.F32, 0x20, 0x30, _lib.BF16, 3, None, 2, _lib.F32,
                                        1, 16, 16, 32, 128, 128, 0) == 0
    for handles in ([good, kv, bad], [good, kv, C.c_void_p(None)]):
        arr = (C.c_void_p * 3)(*[h.value for h in handles])
        rc = lib.dflash_restore_target_cache_after_acceptance(C.cast(arr, _lib.vpp), 3, None, 104, 3, 15, None)
        assert rc == _lib.INVALID
        assert lib.dflash_cache_is_armed(good) and lib.dflash_cache_get_slot(good, 1) == 0x4000
        assert lib.dflash_cache_offset(kv) == 116
        assert lib.dflash_cache_is_armed(bad) and lib.dflash_cache_get_slot(bad, 1) == 0x2000
    for h in (good, kv, bad):
        lib.dflash_cache_destroy(h)


def test_snapshot_cache_restores_pointers():
    lib = _lib.load()
    c = _cache(_lib.CACHE_SNAPSHOT)
    lib.dflash_cache_set_slot(c, 0, 0x1000)
    lib.dflash_cache_set_slot(c, 1, 0x2000)
    lib.dflash_cache_arm_rollback(c, 0)
    assert lib.dflash_cache_record_tape(c, 0x10, 0, 0x20, 0x30, 1, 3, None, 2, 0, 1, 16, 16, 32, 128, 128, 0) == 0
    lib.dflash_cache_set_slot(c, 0, 0x3000)
    lib.dflash_cache_set_slot(c, 1, 0x4000)
    assert lib.dflash_cache_rollback(c, None, 5) == 0
    assert lib.dflash_cache_get_slot(c, 0) == 0x1000 and lib.dflash_cache_get_slot(c, 1) == 0x2000
    lib.dflash_cache_destroy(c)


def test_trim_semantics():
    lib = _lib.load()
    c = _cache(_lib.CACHE_KV)
    lib.dflash_cache_set_offset(c, 5)
    assert lib.dflash_cache_trim(c, 8) == 5 and lib.dflash_cache_offset(c) == 0
    lib.dflash_cache_set_offset(c, 20)
    assert lib.dflash_cache_trim(c, 8) == 8 and lib.dflash_cache_offset(c) == 12
    assert lib.dflash_cache_arm_rollback(c, 0) == _lib.INVALID
    lib.dflash_cache_destroy(c)


@pytest.mark.parametrize("acc,drafted", [(15, 15), (3, 15), (0, 15), (0, 0)])
def test_restore_matches_oracle_actions(acc, drafted):
    """Offsets and armed flags after restoreTargetCacheAfterAcceptance follow the
    oracle's action list (DFlashRuntime.swift:188-223).  No tape is recorded, so no
    kernel is launched."""
    lib = _lib.load()
    kinds = [_lib.CACHE_TAPE, _lib.CACHE_KV, _lib.CACHE_MAMBA, _lib.CACHE_KV, _lib.CACHE_SNAPSHOT]
    names = {_lib.CACHE_TAPE: "rollback", _lib.CACHE_SNAPSHOT: "rollback", _lib.CACHE_MAMBA: "mamba",
             _lib.CACHE_KV: "kv"}
    offsets = [0, 116, 90, 100, 0]
    target_len = 100 + acc + 1
    hs = [_cache(k) for k in kinds]
    for h, k, off in zip(hs, kinds, offsets):
        lib.dflash_cache_set_offset(h, off)
        if k in (_lib.CACHE_TAPE, _lib.CACHE_SNAPSHOT):
            lib.dflash_cache_set_slot(h, 1, 0x2000)
            lib.dflash_cache_arm_rollback(h, 100)
            lib.dflash_cache_set_slot(h, 1, 0x4000)
    arr = (C.c_void_p * len(hs))(*[h.value for h in hs])
    ns = C.c_int64(-1)
    rc = lib.dflash_restore_target_cache_after_acceptance(C.cast(arr, _lib.vpp), len(hs), None, target_len, acc,
                                                          drafted, C.byref(ns))
    assert rc == 0 and ns.value >= 0
    want = O.restore_target_cache_after_acceptance([(names[k], o) for k, o in zip(kinds, offsets)], target_len, acc,
                                                   drafted)
    for h, k, off, action in zip(hs, kinds, offsets, want):
        if action[0] == "clear":
            assert not lib.dflash_cache_is_armed(h)
            assert lib.dflash_cache_get_slot(h, 1) == 0x4000          # keeps the verify forward's state
        elif action[0] == "rollback":
            assert not lib.dflash_cache_is_armed(h)
            assert lib.dflash_cache_get_slot(h, 1) == 0x2000          # snapshot restored (no tape recorded)
        elif action[0] == "set_offset":
            assert lib.dflash_cache_offset(h) == action[1]
        elif action[0] == "trim":
            assert lib.dflash_cache_offset(h) == off - action[1] == target_len
        else:
            assert lib.dflash_cache_offset(h) == off
        lib.dflash_cache_destroy(h)


@pytest.fixture(scope="module")
def rollback_check(tmp_path_factory):
    """Runs tests/rollback/rollback_check.cpp: (launches, status, [(armed, window, state)] per cache)."""
    import subprocess

    exe, lib = tmp_path_factory.mktemp("rollback") / "rollback_check", os.path.dirname(_lib.LIB_PATH)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-rdynamic", os.path.join(ROOT, "tests", "rollback", "rollback_check.cpp"),
                           "-o", str(exe), "-L" + lib, "-ldflash_hip", "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + lib,
                           "-Wl,-rpath,/opt/rocm/lib"])

    def run(refuse, keep, channels, *dks):
        lines = subprocess.run([str(exe)] + [str(x) for x in (refuse, keep, channels, *dks)], capture_output=True, text=True,
                               check=True).stdout.splitlines()
        at = next(i for i, line in enumerate(lines) if line.startswith("status"))
        return lines[:at], int(lines[at].split()[1]), [(int(a), int(w, 16), int(s, 16)) for a, w, s in (line.split() for line in lines[at + 1:])]

    return run


BEFORE, AFTER = (0, 0x100000, 0x300000), (0, 0x500000, 0x700000)      # disarmed, window and state of before and after the verify step


@pytest.mark.parametrize("keep,channels,dks,launches,after", [
    (3, 64, (64, 128), ["replay+windows 1", "replay+windows 1"], AFTER),
    (3, 64, (64, 64, 128), ["replay+windows 2", "replay+windows 1"], AFTER),
    (3, 12, (64, 128), ["replay 1", "replay 1", "windows 2"], AFTER),           # rows of 24 bytes: windows in a launch of their own
    (65535, 8, (64,), ["replay+windows 1"], AFTER),
    (65536, 8, (64,), ["replay 1", "windows 1"], AFTER),                        # more rows than the windows' kernel takes: its refusal
    (3, 0, (64, 128), ["replay 1", "replay 1"], (0, 0x100000, 0x700000)),       # no qkv: the restored window stays
])
def test_rollback_refused_at_any_launch_keeps_both_halves_of_a_cache(rollback_check, keep, channels, dks, launches, after):
    """A rollback takes a launch per replay shape, and any of them may be refused (a head dim that the replay does not take, rows that
    the windows' kernel does not): whichever it is, every cache has the window and the state of the same moment afterwards, those of
    before the verify step, and nothing behind it is launched.  With all of them enqueued both are what the launches write."""
    assert rollback_check(-1, keep, channels, *dks) == (launches, 0, [after] * len(dks))
    for i in range(len(launches)):
        want = launches[:i] + [launches[i] + " refused"]
        assert rollback_check(i, keep, channels, *dks) == (want, _lib.UNSUPPORTED, [BEFORE] * len(dks))


def test_argument_validation_needs_no_gpu_for_null_checks():
    # Null handles are rejected before anything touches a device.
    lib = _lib.load()
    assert lib.dflash_cache_rollback(None, None, 0) == _lib.INVALID
    assert lib.dflash_cache_set_slot(None, 0, None) == _lib.INVALID
    assert lib.dflash_restore_target_cache_after_acceptance(None, 3, None, 0, 0, 0, None) == _lib.INVALID


def test_bench_refuses_more_than_one_gpu():
    """bench.py measures one GPU; asked for more it says so and exits non-zero without touching a device."""
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert r.returncode != 0
    assert "one GPU" in (r.stdout + r.stderr)


def test_ragged_shares_are_found_in_few_sums(tmp_path):
    """How many tiles a workgroup of a ragged attention batch takes: the smallest number that leaves enough workgroups, found by
    halving (at most 2 + log2 of the range), also where a search one by one takes hundreds of sums; tile counts up to 2^20."""
    import math
    import random
    import subprocess

    exe = tmp_path / "shares_check"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", os.path.join(ROOT, "tests", "shares", "shares_check.cpp"), "-o", str(exe)])
    rng = random.Random(0)
    sets = [(2, [3200] + [2600] * 15), (2, [512 + 32 * i for i in range(16)]), (2, [1] * 63 + [3200]), (2, [1, 1]), (64, [300, 1, 7]),
            (255, [1 << 19, (1 << 20) - 1]), (2, [(1 << 18) - i for i in range(64)])]
    for _ in range(400):
        top = rng.choice([8, 300, 3200, 1 << 18])
        sets.append((rng.choice([2, 2, 3, 4, 8, 32, 128]), [rng.randint(1, top) for _ in range(rng.randint(2, 64))]))
    text = "".join(f"{len(t)} {s} {' '.join(map(str, t))}\n" for s, t in sets)
    lines = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.split("\n")
    slowest = 0
    for (s, tiles), line in zip(sets, lines):
        _, sums, linear = map(int, line.split())
        assert sums <= 2 + math.log2(max(tiles)), (s, tiles)
        slowest = max(slowest, linear)
    assert slowest > 200


def _kernel_registers(tmp_path):
    """{kernel name: (vector registers, bytes of scratch)} of the built library's device code."""
    import glob
    import subprocess

    os.symlink(_lib.LIB_PATH, tmp_path / "lib.so")
    subprocess.run(["/opt/rocm/llvm/bin/llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    found = {}
    for f in glob.glob(str(tmp_path / "lib.so.*gfx950")):
        notes = subprocess.run(["/opt/rocm/llvm/bin/llvm-readelf", "--notes", f], capture_output=True, text=True, check=True).stdout
        for entry in notes.split("  - .agpr_count:")[1:]:
            field = lambda name: re.search(r"\.%s:\s+(\S+)" % name, entry).group(1)
            found[field("name")] = int(field("vgpr_count")), int(field("private_segment_fixed_size"))
    return found


@pytest.mark.parametrize("Dk", [64, 128])
@pytest.mark.parametrize("masked", [0, 1])
def test_two_workgroups_of_a_prompt_share_a_compute_unit(tmp_path, Dk, masked):
    """Eight waves each: four waves on a SIMD, which share its 512 registers, and no state in scratch."""
    registers, scratch = next(v for n, v in _kernel_registers(tmp_path).items() if f"gated_delta_long_kernelILi{Dk}ELb{masked}E" in n)
    assert registers <= 128 and scratch == 0


def test_library_builds_without_python():
    """The library and its plain-C clients are what `make` builds by default, on a machine without Python or PyTorch too; the
    Python package's binding is a target of its own."""
    import subprocess

    make = ["make", "-n", "-B", "-C", os.path.join(ROOT, "swiftlm_amd", "csrc"), "PYTHON=/nonexistent"]
    r = subprocess.run(make, capture_output=True, text=True)
    assert r.returncode == 0 and not r.stderr, r.stderr
    assert "libdflash_hip.so" in r.stdout and "step_check" in r.stdout and "_native.so" not in r.stdout
    assert "_native.so" in subprocess.run(make[:-1] + ["native"], capture_output=True, text=True).stdout
