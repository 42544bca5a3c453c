"""Contracts that hold without a GPU: the bench refuses more than one GPU, the product has no CPU fallback, and nothing
outside tests/, the smoke entry and the bench's CPU-baseline leg touches the oracle."""
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_bench_refuses_more_than_one_gpu():
    out = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True, cwd=ROOT)
    assert out.returncode != 0
    assert "--gpus must be 1" in out.stderr
    assert out.stdout.strip() == ""


def test_missing_library_is_an_error_not_a_fallback(monkeypatch, tmp_path):
    from zllm_amd import capi

    monkeypatch.setattr(capi, "_lib", None)
    monkeypatch.setattr(capi, "LIB_PATH", str(tmp_path / "libzllm_attn.so"))
    with pytest.raises(FileNotFoundError, match="no CPU fallback"):
        capi.load()


def test_product_code_does_not_use_the_oracle():
    """Only tests/, __graft_entry__.smoke() and the benches' cpu_baseline leg may import or link anything under oracle/."""
    offenders = []
    for folder, _, files in os.walk(os.path.join(ROOT, "zllm_amd")):
        for name in files:
            if not name.endswith((".py", ".hip", ".hpp", ".cpp", ".h")):
                continue
            path = os.path.join(folder, name)
            text = open(path, encoding="utf-8", errors="replace").read()
            for number, line in enumerate(text.splitlines(), 1):
                if re.search(r"^\s*(import oracle|from oracle)\b|zllm_oracle|oracle/", line):
                    offenders.append((os.path.relpath(path, ROOT), number, line.strip()))
    # the build script links the host layer's parity driver (a test) against the oracle; nothing else may name it
    allowed = {"zllm_amd/build.py"}
    assert [o for o in offenders if o[0] not in allowed] == []
    assert "oracle_dir" in open(os.path.join(ROOT, "zllm_amd", "build.py")).read()


def test_the_probe_kernels_are_not_part_of_the_library():
    """bench.py's plain-read kernels live in their own shared object; the drop-in ABI exports no measurement aid."""
    header = open(os.path.join(ROOT, "include", "zllm_attn.h")).read()
    assert "probe" not in header
    for folder, _, files in os.walk(os.path.join(ROOT, "zllm_amd")):
        for name in files:
            if name.endswith((".py", ".hip", ".hpp", ".cpp", ".h")):
                assert "stream_read" not in open(os.path.join(folder, name), encoding="utf-8", errors="replace").read(), name


def test_a_refused_preferred_workspace_falls_back_to_the_least(monkeypatch):
    """Argument blocks for chunks whose preferred workspace the device has no room for carry the least one; where that is refused too, the
    error is the allocator's."""
    import ctypes as C

    import torch

    from zllm_amd import capi, ops

    lib, empty = capi.load(), torch.empty
    room = [0]

    def limited(size, **kw):
        if size > room[0]:
            raise torch.OutOfMemoryError("no room")
        return empty(size, **kw)

    monkeypatch.setattr(torch, "empty", limited)
    rows, byte = 2048, torch.zeros(1, dtype=torch.uint8)
    q = torch.zeros(rows, 8 * 128, dtype=torch.bfloat16)
    mla_q = torch.zeros(512, 16 * 192, dtype=torch.bfloat16)
    table = torch.zeros(2000, dtype=torch.int32)

    def gqa():
        return ops.gqa_prefill_chunk_args(q, byte, byte, byte, byte, table, 20000, 8, 1, 128, 16, 0.1)

    def mla():
        return ops.mla_decode_args(mla_q, byte, byte, byte, byte, table[None], byte, 16, 192, 256, 512, 64, 64, 4000, query_rows=512)

    for build, least_of, preferred_of in ((gqa, lib.zllm_attn_gqa_prefill_workspace_bytes, lib.zllm_attn_gqa_prefill_preferred_bytes),
                                          (mla, lib.zllm_attn_mla_decode_workspace_bytes, lib.zllm_attn_mla_decode_preferred_bytes)):
        room[0] = 1 << 40
        args, _, workspace = build()
        least, preferred = max(least_of(C.byref(args)), 256), preferred_of(C.byref(args))
        assert args.workspace_bytes == workspace.numel() == preferred > least
        room[0] = preferred - 1
        args, _, workspace = build()
        assert args.workspace_bytes == workspace.numel() == least and args.workspace == workspace.data_ptr()
        room[0] = least - 1
        with pytest.raises(torch.OutOfMemoryError):
            build()
