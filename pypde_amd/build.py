"""Builds libpypde_hip.so in-tree (pypde_amd/_lib/) and checks that the HIP
kernel source compiles for gfx950 through hipRTC.

    python -m pypde_amd.build            # library + kernel compile check
    python -m pypde_amd.build --warm     # also pre-compile the configurations
                                         # used by tests/bench into _lib/_jitcache
"""
import os
import subprocess
import sys
import time

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
LIB = os.path.join(PKG, "_lib", "libpypde_hip.so")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

EMBED = [("PRELUDE_SRC", os.path.join(PKG, "systems", "pde_prelude.h")),
         ("COMMON_SRC", os.path.join(CSRC, "kernels", "ader_common.h")),
         ("WIDE_SRC", os.path.join(CSRC, "kernels", "ader_wide.h")),
         ("WIDE_PRED_SRC", os.path.join(CSRC, "kernels", "ader_wide_predictor.h")),
         ("KERNELS_SRC", os.path.join(CSRC, "kernels", "ader_kernels.h")),
         ("STEP_SRC", os.path.join(CSRC, "kernels", "ader_step.h")),
         ("MLP_SRC", os.path.join(CSRC, "kernels", "mlp_train.h")),
         ("REAL32_SRC", os.path.join(CSRC, "kernels", "real32.h"))]


GEN = os.path.join(PKG, "_build")  # generated sources (not tracked)


def write_embed():
    os.makedirs(GEN, exist_ok=True)
    out = os.path.join(GEN, "kernels_embed.inc")
    parts = ["// generated by pypde_amd/build.py from csrc/kernels and systems/pde_prelude.h\n"]
    for name, path in EMBED:
        text = open(path).read()
        # split into chunks: string literal length stays modest
        chunks = [text[i:i + 12000] for i in range(0, len(text), 12000)] or [""]
        parts.append(f"static const char {name}[] =\n")
        for ch in chunks:
            assert ")PYPDE\"" not in ch
            parts.append(f'R"PYPDE({ch})PYPDE"\n')
        parts.append(";\n")
    new = "".join(parts)
    if not os.path.exists(out) or open(out).read() != new:
        open(out, "w").write(new)


def build_lib():
    write_embed()
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    cmd = [os.path.join(ROCM, "bin", "hipcc"), "-O2", "-std=c++17", "-fPIC", "-shared",
           "--offload-arch=gfx950",
           "-ffp-contract=off", "-Wall", "-Wno-unused-function", "-Wno-unused-result",
           "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-I", GEN,
           os.path.join(CSRC, "pypde_hip.cpp"), os.path.join(CSRC, "tables.cpp"),
           os.path.join(CSRC, "transfer.cpp"), "-pthread",
           "-o", LIB + ".tmp", "-lhiprtc", "-lamdhip64", "-ldl"]
    subprocess.run(cmd, check=True)
    os.replace(LIB + ".tmp", LIB)


def _compile_one(args):
    cfg, recompile = args
    if recompile:
        os.environ["PYPDE_HIP_RECOMPILE"] = "1"
    else:
        os.environ.pop("PYPDE_HIP_RECOMPILE", None)
    from pypde_amd import _capi
    _capi.compile_only(**cfg)
    return cfg["N"]


def main(argv):
    build_lib()
    from pypde_amd import _capi
    _capi.reload()
    from pypde_amd import systems
    # kernel compile check for gfx950 (hipRTC; no GPU needed): the core
    # configurations are compiled on every call, cached code objects or not;
    # with --warm the remaining ones used by the tests and the bench are
    # compiled where the cache lacks them.  Configurations compile in parallel
    # worker processes, the slowest (most variables) first.
    core = systems.standard_configs(full=False)
    cfgs = systems.standard_configs(full="--warm" in argv)
    keys = [repr(sorted(c.items())) for c in core]
    rest = [c for c in cfgs if repr(sorted(c.items())) not in keys]
    jobs = [(c, True) for c in core] + [(c, False) for c in rest]
    jobs.sort(key=lambda j: -j[0]["V"])
    t_start = time.time() - 2.0
    workers = max(1, min(len(jobs), int(os.environ.get("MAX_JOBS", os.cpu_count() or 1)), 8))
    import multiprocessing as mp
    from concurrent.futures import ProcessPoolExecutor
    with ProcessPoolExecutor(max_workers=workers, mp_context=mp.get_context("spawn")) as ex:
        list(ex.map(_compile_one, jobs))
    _capi.check(_capi.lib().pypde_mlp_compile(), "MLP kernel compile")
    pruned = 0
    if "--warm" in argv:
        # code objects that no configuration compiled or fetched in this run
        # are stale (older kernel sources): every fetch refreshes its file time
        cache = os.path.join(PKG, "_lib", "_jitcache")
        for f in os.listdir(cache) if os.path.isdir(cache) else []:
            p = os.path.join(cache, f)
            if f.endswith(".hsaco") and os.path.getmtime(p) < t_start:
                os.remove(p)
                pruned += 1
    print(f"built {LIB}; hipRTC gfx950 kernels: {len(core)} configurations compiled, "
          f"{len(cfgs)} present, {pruned} stale code objects removed")


if __name__ == "__main__":
    main(sys.argv[1:])
