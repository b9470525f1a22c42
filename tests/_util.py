"""Shared helpers for the parity tests: tensor conversion and error statistics."""

from __future__ import annotations

import ctypes

import numpy as np
import torch

from oracle.numerics import bf16_ulp


def to_np(t: torch.Tensor) -> np.ndarray:
    """Any torch tensor (bf16 included) -> float32 numpy array on the host (exact for bf16)."""
    return t.detach().to("cpu", torch.float32).numpy()


def ulp_stats(got: np.ndarray, want: np.ndarray) -> dict:
    """Elementwise differences measured in bf16 ulps of the expected value."""
    got = np.asarray(got, np.float32)
    want = np.asarray(want, np.float32)
    diff = np.abs(got.astype(np.float64) - want.astype(np.float64))
    ulps = diff / bf16_ulp(want).astype(np.float64)
    return {
        "max_ulps": float(ulps.max()) if ulps.size else 0.0,
        "mismatch": float(np.mean(diff > 0)) if diff.size else 0.0,
        "max_abs": float(diff.max()) if diff.size else 0.0,
    }


def abs_stats(got: np.ndarray, want: np.ndarray) -> dict:
    diff = np.abs(np.asarray(got, np.float64) - np.asarray(want, np.float64))
    return {"max_abs": float(diff.max()), "mean_abs": float(diff.mean())}


def describe(label: str, stats: dict) -> str:
    return label + " " + " ".join(f"{k}={v:.3g}" for k, v in stats.items())


class _KernelNodeParams(ctypes.Structure):
    """hipKernelNodeParams (hip_runtime_api.h)."""
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", ctypes.c_uint * 3), ("params", ctypes.c_void_p), ("shared", ctypes.c_uint)]


def _kernel_nodes(fn) -> list:
    """(grid, name) of every kernel that ``fn`` launches, read from a captured graph."""
    from flicker_amd import _lib
    hip = _lib.lib()   # its symbols include those of the HIP runtime it is linked to
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        fn()
    raw, count = ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(count)) == 0
    nodes = (ctypes.c_void_p * max(1, count.value))()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(count)) == 0
    found = []
    for node in nodes[:count.value]:
        kind, p = ctypes.c_int(-1), _KernelNodeParams()
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        if kind.value == 0:   # hipGraphNodeTypeKernel
            assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
            found.append((tuple(p.grid), hip.hipKernelNameRefByPtr(ctypes.c_void_p(p.func), None).decode()))
    return found


def launches(fn) -> list:
    """The grid (x, y, z) of every kernel that ``fn`` launches."""
    return [grid for grid, _ in _kernel_nodes(fn)]


def kernel_names(fn) -> list:
    """The (mangled) name of every kernel that ``fn`` launches."""
    return [name for _, name in _kernel_nodes(fn)]
