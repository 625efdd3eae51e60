"""The C-ABI library loads and exports every entry point the header declares."""

from __future__ import annotations

import re
from pathlib import Path

import pytest

from opake_amd import _native

HEADER = Path(__file__).resolve().parents[1] / "include" / "opake_amd.h"


def declared_functions() -> set[str]:
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return set(re.findall(r"\b(dpc_[a-z0-9_]+)\s*\(", text))


def test_header_declares_the_bound_functions():
    assert declared_functions() == set(_native.SIGNATURES)


def test_library_exports_every_declared_symbol():
    if not _native.LIB_PATH.exists():
        pytest.skip("native library not built")
    lib = _native.load()
    for name in declared_functions():
        assert hasattr(lib, name), name


def test_version_and_size_queries():
    if not _native.LIB_PATH.exists():
        pytest.skip("native library not built")
    lib = _native.load()
    assert lib.dpc_version() == _native.ABI_VERSION == 207
    assert lib.dpc_clip_plan_bytes(32) == 16 + 32 * 4
    # Grouped Gram workspace: the records, then the split kernel's tickets and
    # accumulator exchange (2 x 224 KiB per set), each 256-byte aligned.
    assert lib.dpc_grouped_gram_workspace_bytes(10, 0) == 1024
    assert lib.dpc_grouped_gram_workspace_bytes(10, 3) == 1024 + 256 + 3 * 2 * 229376
    assert lib.dpc_gram_workspace_bytes(0, 5) == 0
    assert lib.dpc_gram_workspace_bytes(2, 128) > 0


def test_gram_workspace_of_a_layer():
    """Only layers off the bf16 MFMA path are given records of 32-row tile pairs (12
    float64 words each): the others keep to those of 64 rows, and two words an example."""
    if not _native.LIB_PATH.exists():
        pytest.skip("native library not built")
    lib = _native.load()

    def query(B, T, din, dout, dtype, bias=0):
        return lib.dpc_gram_layer_workspace_bytes(B, T, din, dout, dtype, bias)

    def records(B, T, rows):
        n = -(-T // rows)
        return n * (n + 1) // 2 * B * 96

    def up(n):
        return -(-n // 256) * 256

    f32, bf16 = _native.DPC_F32, _native.DPC_BF16
    for B, T in ((8, 300), (4, 4160), (2, 32640)):  # odd numbers of 128-row blocks
        assert query(B, T, 4096, 4096, bf16) == up(records(B, T, 64) + 16 * B)
        assert query(B, T, 4096, 4096, bf16, 1) == up(records(B, T, 64) + 16 * B) + 256 * B
    assert query(8, 300, 4096, 4096, f32) == up(records(8, 300, 32))
    assert query(8, 300, 4095, 4096, bf16) == up(records(8, 300, 32))
    assert query(8, 4160, 4096, 4096, f32) == up(records(8, 4160, 64) + 128)
    # A biased layer of the one-launch path also holds its counters.
    assert (query(6, 256, 128, 264, bf16, 1)
            == up(query(6, 256, 128, 264, bf16) + 6 * 256) + lib.dpc_gram_clip_counter_bytes(6, 256))
    # The queries without a layer hold any of them.
    for B, T, din, dout, dtype, bias in ((6, 256, 128, 264, bf16, 1), (8, 300, 4096, 4096, f32, 1),
                                         (8, 4160, 33, 9, bf16, 1), (1, 70, 8, 8, f32, 0)):
        assert query(B, T, din, dout, dtype, bias) <= lib.dpc_gram_clip_workspace_bytes(B, T)
        assert query(B, T, din, dout, dtype) <= lib.dpc_gram_workspace_bytes(B, T)


def test_clipped_sum_workspace_of_huge_odd_outputs():
    """Odd output rows of the bf16 MFMA path are finished by a launch of a thread per 2 x 2
    values: outputs of more than it covers (2^32 threads) keep to the generic path, which
    needs no float32 plane of the output."""
    if not _native.LIB_PATH.exists():
        pytest.skip("native library not built")
    lib = _native.load()
    bias = 32 * 131072 * 4
    assert lib.dpc_clipped_sum_workspace_bytes(2, 64, 131073, 131072, _native.DPC_BF16) == bias
    plane = 131072 * 65544 * 4
    assert lib.dpc_clipped_sum_workspace_bytes(2, 64, 65537, 131072, _native.DPC_BF16) > plane


def test_tables_used_under_keep_alive_survive_eviction():
    # A graph owner holds the tables its capture used: filling the content
    # cache past its bound afterwards evicts the cache's entries but not the
    # owner's references (CPU tables: the cache logic is device-independent).
    import gc
    import weakref

    from opake_amd import _tables

    with _tables.keep_alive() as kept:
        t1 = _tables.device_table([1, 2, 3], "int32", "cpu")
        t2 = _tables.device_table([1, 2, 3], "int32", "cpu")  # a cache hit
    assert t1 is t2 and any(x is t1 for x in kept)
    ref = weakref.ref(t1)
    del t1, t2
    for i in range(_tables._MAX_ENTRIES + 10):
        _tables.device_table([i, i + 1, 7777], "int32", "cpu")
    gc.collect()
    assert ref() is not None  # evicted from the cache, alive through `kept`
    del kept
    gc.collect()
    assert ref() is None


def test_err_less_accumulation_must_be_explicit():
    # Accumulating norms into `out` without `err` drops the bound of the sum;
    # the norm helpers refuse it unless return_error=False says so.
    from opake_amd import ops
    from opake_amd.exceptions import ConfigurationError

    out, err = object(), object()
    assert ops._wants_error(None, None, None) is False
    assert ops._wants_error(None, None, True) is True
    assert ops._wants_error(out, err, None) is True
    assert ops._wants_error(out, None, False) is False
    with pytest.raises(ConfigurationError, match="drops the rounding-error bound"):
        ops._wants_error(out, None, None)
    with pytest.raises(ConfigurationError, match="return_error=False"):
        ops._wants_error(out, err, False)


def _kernarg_setting(env_value):
    """HIP_FORCE_DEV_KERNARG as seen after `import opake_amd` in a fresh
    interpreter whose environment holds `env_value` (None: unset)."""
    import os
    import subprocess
    import sys

    env = {k: v for k, v in os.environ.items() if k != "HIP_FORCE_DEV_KERNARG"}
    if env_value is not None:
        env["HIP_FORCE_DEV_KERNARG"] = env_value
    code = "import os, opake_amd; print(os.environ.get('HIP_FORCE_DEV_KERNARG'))"
    out = subprocess.run([sys.executable, "-c", code], env=env, check=True, text=True,
                         capture_output=True, cwd=Path(__file__).resolve().parents[1])
    return out.stdout.strip()


def test_import_asks_for_device_kernel_arguments_unless_set():
    assert _kernarg_setting(None) == "1"
    assert _kernarg_setting("0") == "0"
