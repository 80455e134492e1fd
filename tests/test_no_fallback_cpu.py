"""The product path has no CPU fallback: without the built library every entry raises, and CPU
tensors are rejected before any native call (CPU tests; nothing here launches a kernel)."""

import pathlib
import subprocess
import sys
import textwrap

import pytest
import torch

from lastkv_amd import ops

REPO = pathlib.Path(__file__).resolve().parents[1]


def test_missing_library_raises_native_error():
    # a fresh process whose library path names nothing: load() and the ops built on it must raise
    code = textwrap.dedent(
        """
        import pathlib, sys
        sys.path.insert(0, sys.argv[1])
        from lastkv_amd import _lib, ops
        _lib.LIB_PATH = pathlib.Path(sys.argv[1]) / "no_such_dir" / "liblastkv_amd.so"
        for call in (_lib.load, lambda: ops.decode_workspace_bytes(1, 8, 1)):
            try:
                call()
            except _lib.LastKVNativeError as e:
                assert "is not built" in str(e), e
            else:
                raise SystemExit("no error without the library")
        print("ok")
        """
    )
    proc = subprocess.run([sys.executable, "-c", code, str(REPO)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0 and proc.stdout.strip() == "ok", proc.stdout + proc.stderr


def test_cpu_tensors_are_rejected():
    B, Hq, Hkv, D = 1, 8, 2, 128
    q = torch.zeros(B, Hq, D, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="GPU"):
        ops.decode_attention(q, local=ops.TiledKV.zeros(B, Hkv, 64, "cpu"), local_len=1)


def test_without_the_launch_module_the_python_bodies_make_the_calls():
    # a process in which lastkv_amd._host cannot be imported: the library still loads, every hot op reaches its
    # Python body (whose first check refuses the CPU tensors) and nothing asks for the module
    code = textwrap.dedent(
        """
        import sys
        sys.path.insert(0, sys.argv[1])
        sys.modules["lastkv_amd._host"] = None  # (import raises ImportError)
        import torch
        from lastkv_amd import _lib, ops
        assert ops._host is None and _lib.load() is not None
        x = torch.zeros(2, 64, dtype=torch.bfloat16)
        q = torch.zeros(1, 8, 128, dtype=torch.bfloat16)
        rows = dict(num_q_heads=8, num_kv_heads=2, q_norm_weight=None, k_norm_weight=None, eps=1e-5, positions=0, ring=None)
        for call in (lambda: ops.rmsnorm(x, x[0], 1e-5), lambda: ops.silu_mul(x, x), lambda: ops.decode_attention(q),
                     lambda: ops.prefill_attention(q[None]), lambda: ops.qkv_epilogue(q, q, q, q, q, **rows)):
            try:
                call()
            except ValueError as e:
                assert "GPU" in str(e), e
            else:
                raise SystemExit("no error for CPU tensors")
        print("ok")
        """
    )
    proc = subprocess.run([sys.executable, "-c", code, str(REPO)], capture_output=True, text=True, timeout=300)
    assert proc.returncode == 0 and proc.stdout.strip() == "ok", proc.stdout + proc.stderr
