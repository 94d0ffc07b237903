"""The C-ABI library loads on a CPU-only host and exports every symbol the header declares."""
import ctypes
import re
from pathlib import Path

import pytest

from piper_amd import _lib

HEADER = Path(__file__).resolve().parents[1] / "include" / "piper_amd.h"


def declared_symbols():
    text = HEADER.read_text()
    return sorted(set(re.findall(r"^PK_API\s+[\w\s\*]+?\b(pk_\w+)\s*\(", text, flags=re.M)))


def test_header_declares_the_expected_entry_points():
    syms = declared_symbols()
    assert len(syms) >= 21
    for must in ("pk_route_topk", "pk_sort_by_expert", "pk_permute_fwd", "pk_combine_fwd",
                 "pk_grouped_swiglu_fwd", "pk_grouped_swiglu_dgrad", "pk_grouped_swiglu_wgrad",
                 "pk_bucket_plan", "pk_bucket_pack", "pk_adamw_fused"):
        assert must in syms


def test_library_exports_every_declared_symbol():
    assert _lib.is_built(), "build the library first: python -m piper_amd.build"
    lib = ctypes.CDLL(str(_lib.LIB_PATH))
    for name in declared_symbols():
        assert hasattr(lib, name), f"{name} declared in the header but not exported"
    # and the ctypes signature table covers exactly the declared set
    assert sorted(_lib.SIGNATURES) == declared_symbols()


def test_host_only_calls():
    lib = _lib.load()
    assert lib.pk_version() >= 100
    assert _lib.status_string(0) == "ok"
    assert "argument" in _lib.status_string(-1)
    assert lib.pk_sort_workspace_bytes(32768, 128) == (32768 // 512) * 128 * 4
    assert lib.pk_sort_workspace_bytes(-1, 128) < 0


def test_decode_step_refuses_what_the_norm_refuses():
    """A negative or undefined eps is an argument error in pk_rmsnorm_fwd, and in the calls that have the norm in them (the
    check comes before any launch; without a norm eps is not looked at, and the workspace check is next)."""
    lib = _lib.load()
    buf = ctypes.create_string_buffer(1 << 16)
    p = (ctypes.addressof(buf) + 15) // 16 * 16
    T, H, E, I, K = 1, 64, 4, 64, 2

    def decode(norm_w, eps):
        return lib.pk_region_decode(p, _lib.PK_BF16, norm_w, eps, p, None, p, p, p, 1, 1.0, None, p, T, H, E, I, K, None, 0, None)

    workspace = decode(p, 1e-6)
    assert "workspace" in _lib.status_string(workspace) and decode(None, -1.0) == workspace
    for eps in (-1e-6, float("nan"), float("-inf")):
        norm = lib.pk_rmsnorm_fwd(p, _lib.PK_BF16, p, eps, p, None, T, H, None)
        assert "invalid argument" in _lib.status_string(norm)
        assert decode(p, eps) == norm
        assert lib.pk_norm_gate_route_sort(p, _lib.PK_BF16, p, eps, p, None, p, None, T, H, E, K, 1, 1.0, p, p, p, None, p, p, None, None, p, 0,
                                           None) == norm


def test_decode_step_pays_only_where_it_applies():
    lib = _lib.load()
    for T in (-1, 0, 1, 2, 5, 16, 17, 2**62):
        for K in (0, 1, 4, 16, 17, 2**62):
            for H, E, I in ((256, 16, 128), (2048, 128, 768), (8192, 64, 1024), (1000, 24, 360)):
                if lib.pk_region_decode_pays(T, H, E, I, K):
                    assert T > 0 and 0 < T * K <= 16
                    assert K > E or lib.pk_region_decode_workspace_bytes(T, H, E, I, K, _lib.PK_BF16) > 0


def test_counter_sets_are_handed_out_per_stream_and_capture():
    """Launches that can overlap must not share scheduling counters: every (stream, capture
    sequence) pair keeps a set of its own; the same pair always gets the same set."""
    lib = _lib.load()
    dev = 63                      # a device index no GPU test uses: the directory starts empty there
    stream_a, stream_b = 0x7f0000001000, 0x7f0000002000
    a = lib.pk_sched_slot_index(dev, stream_a, 0, 0)
    b = lib.pk_sched_slot_index(dev, stream_b, 0, 0)
    assert a >= 0 and b >= 0 and a != b
    assert lib.pk_sched_slot_index(dev, stream_a, 0, 0) == a          # stable per stream
    # a launch recorded into a graph on stream a: another set than eager work on stream a,
    # and another capture another set again
    g1 = lib.pk_sched_slot_index(dev, stream_a, 1, 0)
    g2 = lib.pk_sched_slot_index(dev, stream_a, 2, 0)
    assert len({a, b, g1, g2}) == 4
    assert lib.pk_sched_slot_index(dev, stream_a, 1, 0) == g1
    # the per-thread default stream is one handle for many streams: the thread is part of the key
    t1 = lib.pk_sched_slot_index(dev, 2, 0, 111)
    t2 = lib.pk_sched_slot_index(dev, 2, 0, 222)
    assert t1 != t2 and len({a, b, g1, g2, t1, t2}) == 6
    # the null stream has a set like any other
    assert lib.pk_sched_slot_index(dev, 0, 0, 0) not in {a, b, g1, g2, t1, t2}
    # more keys than sets: shared round-robin, still a valid index, and old keys keep theirs
    seen = {lib.pk_sched_slot_index(dev, 0x100000 + 64 * i, 0, 0) for i in range(1100)}
    assert all(0 <= s < 1024 for s in seen) and len(seen) == 1024
    assert lib.pk_sched_slot_index(dev, stream_a, 0, 0) == a
    assert lib.pk_sched_slot_index(-1, 0, 0, 0) < 0 and lib.pk_sched_slot_index(64, 0, 0, 0) < 0


def test_the_scaled_backward_in_units_of_more_than_128_rows_does_not_compile(tmp_path):
    """Its epilogue would store through outputs that are null where only the transposed copies are read."""
    import shutil
    import subprocess
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(hipcc).exists():
        pytest.skip("no hipcc")
    src = Path(_lib.__file__).resolve().parent / "csrc" / "grouped_gemm.hip"
    for epilogue, compiles in (("EPI_SWIGLU_BWD", True), ("EPI_SWIGLU_BWD_SCALED", False)):
        unit = tmp_path / f"{epilogue}.hip"
        unit.write_text(f'#include "{src}"\nnamespace {{ template __global__ void mf::ragged_m_kernel<256, 256, 32, 2, 4, 4, false, mf::{epilogue}>'
                        "(const mf::RaggedMParams); }\n")
        run = subprocess.run([hipcc, "--offload-arch=gfx950", "-std=c++17", "--cuda-device-only", "-fsyntax-only", str(unit)],
                             capture_output=True, text=True, timeout=120)
        assert (run.returncode == 0) == compiles, run.stderr
        assert compiles or "the unscaled backward only" in run.stderr, run.stderr
