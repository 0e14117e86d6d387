"""Builds libmfmoe.so (the HIP kernels + C ABI) in-tree with hipcc for gfx950."""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libmfmoe.so")
SOURCES = ["format.hip", "gemv.hip", "int8_mlp.hip", "router.hip", "router_family.hip", "moe_decode.hip", "moe_fused.hip",
           "moe_prefill.hip", "qmm_ring.hip", "qmm_resident.hip", "qmm_tile32.hip", "static_scratch.hip", "api.hip"]

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-ffp-contract=off",
    # packed-FP32 instructions are switched off for all device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wextra", "-Wno-unused-parameter",
]


SHAPES_JSON = os.path.join(HERE, "fused_shapes.json")
SHAPES_INC = os.path.join(CSRC, "fused_shapes.inc")
_BITS = {4: "kBits4", 2: "kBits2", 1: "kBitsTernary"}
_MF_BITS = {4: "MF_BITS_4", 2: "MF_BITS_2", 1: "MF_BITS_TERNARY"}


def load_shapes(extra: str | None = None) -> list[dict]:
    """The listed layer shapes: fused_shapes.json plus the file MF_FUSED_SHAPES (or `extra`) names."""
    import json
    shapes = list(json.load(open(SHAPES_JSON))["shapes"])
    extra = extra or os.environ.get("MF_FUSED_SHAPES")
    if extra:
        shapes += list(json.load(open(extra))["shapes"])
    seen, out = set(), []
    for sh in shapes:
        key = tuple(sh[k] for k in ("bits", "shared_bits", "d", "f", "num_experts", "top_k", "shared_f", "router_mode", "maple"))
        if sh["bits"] not in _BITS or (sh["shared_f"] and sh["shared_bits"] not in _BITS):
            raise ValueError(f"fused shape {sh.get('name')}: bits must be 4, 2 or 1")
        if sh["d"] % 64 or sh["f"] % 64 or sh["shared_f"] % 64 or not 0 < sh["top_k"] <= 8 or not 0 < sh["num_experts"] <= 512:
            raise ValueError(f"fused shape {sh.get('name')}: sizes out of range")
        if key not in seen:
            seen.add(key)
            out.append(sh)
    return out


def shape_from_arch(arch: dict, bits: int = 4, shared_bits: int = 4, shared_gated: bool = False) -> dict:
    """One entry of the shape list from the architecture block of a model manifest (the reference's ArchConfig,
    Infrastructure/ModelIO/ModelTypes.swift:176-200: hiddenSize, moeIntermediateSize, numExperts, topKExperts;
    intermediateSize is the shared expert's width where the model has a gated shared expert)."""
    return {"name": arch.get("name", "model"), "bits": bits, "shared_bits": shared_bits, "d": int(arch["hiddenSize"]),
            "f": int(arch["moeIntermediateSize"]), "num_experts": int(arch["numExperts"]),
            "top_k": int(arch["topKExperts"]), "shared_f": int(arch["intermediateSize"]) if shared_gated else 0,
            "router_mode": 0, "maple": 0}


def write_shapes_inc(shapes: list[dict]) -> str:
    """csrc/fused_shapes.inc: for every listed shape four instances of the fused decode kernel -- one token row
    (all dimensions and flags literals) and any number of rows (dimensions literals), each with the layer's own
    router and with caller-given routing -- and the branches of the launcher that pick them."""
    decl, own, given = [], [], []
    for i, sh in enumerate(shapes):
        dims = f"{sh['d']}, {sh['f']}, {sh['num_experts']}, {sh['top_k']}"
        fs, mode, maple = sh["shared_f"], sh["router_mode"], sh["maple"]
        b, sb = _BITS[sh["bits"]], _BITS[sh["shared_bits"] if fs else 4]
        decl += [f"// {sh.get('name', 'shape %d' % i)}",
                 f"using Gen{i}T1 = StaticShape<{dims}, 1, {fs}, false, {mode}, {maple}, 1, 1>;",
                 f"using Gen{i}Tn = StaticShape<{dims}, kDyn, {fs}>;",
                 f"using Gen{i}T1Given = StaticShape<{dims}, 1, {fs}, true, kDyn, {maple}, 1, 1>;",
                 f"using Gen{i}TnGiven = StaticShape<{dims}, kDyn, {fs}, true>;"]
        cond = (f"c.bits == {_MF_BITS[sh['bits']]} && c.d == {sh['d']} && c.f == {sh['f']} && "
                f"c.num_experts == {sh['num_experts']} && c.top_k == {sh['top_k']} && c.shared_f == {fs}")
        if fs:
            cond += f" && c.shared_bits == {_MF_BITS[sh['shared_bits']]}"
        one = f"one && c.maple_rounding == {maple}u && no_limit && a.xprep"
        own.append(f"  else if ({cond} && c.router_mode == {mode}) {{\n"
                   f"    if ({one}) MF_FUSED({b}, {sb}, Gen{i}T1);\n    else MF_FUSED({b}, {sb}, Gen{i}Tn);\n  }}")
        given.append(f"  else if ({cond}) {{\n"
                     f"    if ({one}) MF_FUSED({b}, {sb}, Gen{i}T1Given);\n    else MF_FUSED({b}, {sb}, Gen{i}TnGiven);\n  }}")
    text = ("// Generated by mference_amd/build.py from fused_shapes.json (and the file MF_FUSED_SHAPES names): instances of\n"
            "// the fused decode launch for the listed layer shapes.  Included three times by moe_fused.hip, once per section.\n"
            "#if defined(MF_SHAPES_DECLARE)\n" + "\n".join(decl) + "\n"
            "#elif defined(MF_SHAPES_PICK_OWN)\n" + "\n".join(own) + "\n"
            "#elif defined(MF_SHAPES_PICK_GIVEN)\n" + "\n".join(given) + "\n#endif\n")
    if not os.path.exists(SHAPES_INC) or open(SHAPES_INC).read() != text:
        with open(SHAPES_INC, "w") as fh:
            fh.write(text)
    return SHAPES_INC


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        raise RuntimeError("hipcc failed: " + " ".join(cmd[-3:]))
    if verbose and proc.stderr:
        sys.stderr.write(proc.stderr)


def build(verbose: bool = False, only: list[str] | None = None) -> str:
    """Compiles every source to an object of its own (in parallel) and links them.  `only` names the
    sources to recompile when the other objects are already there (a developer's shortcut; the build
    check compiles everything)."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    os.makedirs(OBJ, exist_ok=True)
    write_shapes_inc(load_shapes())
    objs = [os.path.join(OBJ, s.replace(".hip", ".o")) for s in SOURCES]
    if only is not None:
        only = [s if s.endswith(".hip") else s + ".hip" for s in only]
        unknown = [s for s in only if s not in SOURCES]
        if unknown:
            raise ValueError(f"not a source of the library: {unknown}")
    todo = [(s, o) for s, o in zip(SOURCES, objs) if only is None or s in only or not os.path.exists(o)]
    jobs = min(8, max(1, (os.cpu_count() or 2) * 3 // 4))
    with ThreadPoolExecutor(jobs) as pool:
        list(pool.map(lambda so: _run([hipcc, *FLAGS, "-c", "-o", so[1], os.path.join(CSRC, so[0])], verbose), todo))
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs], verbose)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True, only=sys.argv[1:] or None))
