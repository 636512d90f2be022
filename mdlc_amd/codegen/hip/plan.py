"""The launch-plan contract: ``Launch`` records and the ``HipModule``.

Field names follow mdlc/codegen/cuda/emit.py:38-95 (``Launch``,
``CudaModule``): a launch is a kind, a kernel name, its input and output
edges in kernel-argument order, grid, block and a metadata dict.
"""

from __future__ import annotations

from dataclasses import dataclass, field

from mdlc_amd.codegen.hip import templates as T
from mdlc_amd.ir import Graph

LIBRARY_PARTS = ("common", "gemm_f32", "gemm_x3", "conv_x3", "gemm_wsplit", "conv_wino", "conv_wino_x3", "conv_pool",
                 "im2col", "pool", "dwconv", "copy", "layout")
QUANT_OPS = {"QuantizeLinear", "DequantizeLinear", "QConv", "QGemm", "QAdd", "QLut",
             "QGlobalAveragePool", "QMlp"}
# The library parts a launch kind's kernel needs beyond "common" and
# "gemm_f32" (which every module takes: the epilogue helpers and the
# compile-time window types live there). A module compiles only the parts
# its launches use, so a change to one kernel file leaves the code objects of
# modules that do not use it valid.
KIND_PARTS = {"gemm_ws": ("gemm_wsplit",), "conv_ws": ("gemm_wsplit",), "wino": ("conv_wino",),
              "conv_pool": ("conv_pool",),
              "im2col": ("im2col",), "dwconv": ("dwconv",), "maxpool": ("dwconv",),
              "avgpool": ("dwconv",), "gap": ("pool",), "copy": ("copy",), "softmax": ("layout",),
              "transpose": ("layout",), "pad": ("layout",), "concat": ("layout",)}
INT8_KINDS = {"quantize", "qgemm", "qconv_first", "qmlp", "qdwconv", "qadd", "qlut", "qgap",
              "dequantize"}


def library_parts(kinds, more=()) -> tuple:
    """The library parts, in LIBRARY_PARTS order (int8 last), that launches of
    ``kinds`` need, with those of ``more``."""
    need = {"common", "gemm_f32"} | set(more)
    for k in kinds:
        need.update(KIND_PARTS.get(k, ()))
    return tuple(p for p in LIBRARY_PARTS if p in need) + \
        (("int8",) if any(k in INT8_KINDS for k in kinds) else ())


def round16(n: int) -> int:
    return (int(n) + 15) // 16 * 16


def round4(n: int) -> int:
    return (int(n) + 3) // 4 * 4


@dataclass
class Launch:
    """One kernel invocation of the plan (contract of emit.py:38-47)."""
    kind: str
    kernel_name: str
    inputs: list
    outputs: list
    grid: tuple
    block: tuple
    meta: dict = field(default_factory=dict)


@dataclass
class HipModule:
    graph: Graph
    kernels: dict                  # kernel name -> wrapper source
    plan: list                     # [Launch]
    scratch_shapes: dict           # scratch tensor -> (rows, ld) float32
    device_constants: dict = field(default_factory=dict)   # packed constant -> ndarray
    library: tuple = LIBRARY_PARTS
    # scratch tensor -> region class; tensors of one class share one region
    # (they are used strictly one after another on the stream)
    scratch_class: dict = field(default_factory=dict)
    # tensor -> device layout when it differs from the IR's NCHW ("NHWC" for
    # int8 activations); the executor converts when a tensor is read or written
    device_layout: dict = field(default_factory=dict)

    def sources(self) -> str:
        """One hipRTC translation unit: the templates, then every wrapper."""
        head = "// Generated by mdlc_amd for gfx950.\n"
        lib = "\n".join(T.library_source(p) for p in self.library)
        return head + lib + "\n" + "\n".join(self.kernels[k] for k in sorted(self.kernels))

    def fallbacks(self) -> list:
        """Host-executed launches: always empty — every op runs on the device."""
        return [l.kernel_name for l in self.plan if l.kind == "host"]

    def report(self) -> str:
        kinds: dict = {}
        for l in self.plan:
            kinds[l.kind] = kinds.get(l.kind, 0) + 1
        fb = self.fallbacks()
        return "\n".join([
            f"HIP module: {len(self.kernels)} distinct kernels, {len(self.plan)} launches",
            "  launches by kind: " + ", ".join(f"{k}x{v}" for k, v in sorted(kinds.items())),
            "  host fallbacks: " + (", ".join(fb) if fb else "none"),
        ])
