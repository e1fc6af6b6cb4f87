"""Checks on the gfx950 assembly of the kernels (compiled here from source, no GPU needed)."""
import os
import re
import subprocess

from burn_dragon_amd import build


def _device_assembly(tmp_path, sources):
    procs = []
    for src in sources:
        out = str(tmp_path / (src + ".s"))
        cmd = [build.HIPCC, *build.FLAGS, "--offload-device-only", "-S", os.path.join(build.CSRC, src), "-o", out]
        procs.append((out, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    for out, proc in procs:
        log, _ = proc.communicate()
        assert proc.returncode == 0, log
    return [open(out).read() for out, _ in procs]


def test_loads_into_lds_keep_a_wait_state_behind_a_write_of_m0(tmp_path):
    """A load into LDS takes its place from M0; behind a scalar write of M0 it needs one wait state, i.e. any other
    instruction in between.  The compiler sees to that for its own loads, hand-written ones have to do it themselves."""
    sources = [s for s in build.SOURCES
               if re.search(r"load_lds|copy_to_lds|copy_piece_to_lds", open(os.path.join(build.CSRC, s)).read())]
    assert {"attention_parallel.hip", "prefill.hip"} <= set(sources)
    for src, text in zip(sources, _device_assembly(tmp_path, sources)):
        lines = [l.split(";")[0].strip() for l in text.splitlines()]
        code = [l for l in lines if l and not l.startswith(".") and not l.endswith(":")]
        loads = [i for i, l in enumerate(code) if re.match(r"(global_load_lds|(global|buffer)_load.*\blds\b)", l)]
        assert loads, src
        for i in loads:
            assert not re.match(r"s_\w+ m0\b", code[i - 1]), (src, code[i - 1 : i + 1])
