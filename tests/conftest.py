"""Shared pytest setup: the `gpu` marker, repo root on sys.path, the oracle build, the dispatch rules."""
import ctypes
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built libnnq.so")


def _ensure_oracle():
    lib = os.path.join(ROOT, "oracle", "liboracle.so")
    src = os.path.join(ROOT, "oracle", "nnq_oracle.c")
    if not os.path.exists(lib) or os.path.getmtime(lib) < os.path.getmtime(src):
        subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "oracle")], check=True)


_ensure_oracle()


@pytest.fixture(scope="session")
def O():
    from oracle import oracle
    return oracle


@pytest.fixture(scope="session")
def rules():
    """Which kernel a shape takes (nn_amd/csrc/nnq_plan.cpp)."""
    from nn_amd import _lib
    lib = _lib.load()
    i64, c_int = ctypes.c_int64, ctypes.c_int
    lib.nnq_rule_few_rows.argtypes = [c_int, i64, i64, i64, c_int]
    lib.nnq_rule_gemm_wide.argtypes = [i64, i64, i64, c_int, c_int, ctypes.POINTER(c_int)]
    lib.nnq_rule_gemm_wide6.argtypes = [i64, i64, i64]
    lib.nnq_rule_moe_few.argtypes = [i64, i64, i64, i64, c_int, c_int]

    class Rules:
        @staticmethod
        def few_rows(fmt, m, n, k, bf16):
            return lib.nnq_rule_few_rows(fmt, (n + 15) // 16, k, m, bf16)

        @staticmethod
        def wide(m, n, k, bf16, h_out=0):
            """(column tiles per workgroup, K split); (0, 0) where the wide Q4_K kernel does not take it"""
            ks = c_int(0)
            return lib.nnq_rule_gemm_wide(m, n // 16, k // 256, bf16, h_out, ctypes.byref(ks)), ks.value

        @staticmethod
        def wide6(m, n, k):
            return lib.nnq_rule_gemm_wide6(m, n // 16, k // 256)

        @staticmethod
        def moe_few(experts, hidden, inter, tokens, top_k, bf16):
            return lib.nnq_rule_moe_few(experts, hidden, inter, tokens, top_k, bf16)

    return Rules
