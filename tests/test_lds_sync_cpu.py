"""LDS writes are waited for before the barrier that publishes them.

The LDS-DMA kernel's main loop uses a bare s_barrier (no fence, so that its DMA
loads stay in flight), and gfx950 adds no wait of its own: where the loader
stores f(X_upper) to LDS for the other waves to read after the barrier, the
writer has to wait for those stores first.  Checked on the assembly of the
configurations that store from registers, over every path through the code."""
import re
import subprocess

import pytest

from lich_amd import build as B

# operand type, mode, activation, BM, BN, stages, wave rows, wave columns (ipc_s16.hip, ipc_s16_t*.hip)
CONFIGS = {
    "tall_pred": "bf16, S16_PRED, 1, ACT_TANH, true, 512, 64, 2, 8, 1",
    "tiles0_pred": "f16, S16_PRED, 1, ACT_RELU, true, 256, 128, 3, 4, 4",
    "tiles2_weight": "bf16, S16_WEIGHT, 1, ACT_RELU, true, 128, 128, 2, 2, 2",
    "tiles3_fwd": "f16, S16_FWD, 1, ACT_RELU, true, 256, 256, 2, 2, 4",
}


def _unwaited_barriers(body):
    """Barriers that some path reaches with an LDS write not yet waited for (lgkmcnt(0))."""
    lines = [ln.split(";")[0].split("//")[0].strip() for ln in body.splitlines()]
    lines = [ln for ln in lines if ln and (not ln.startswith(".") or ln.endswith(":"))]
    label = {ln[:-1]: i for i, ln in enumerate(lines) if ln.endswith(":")}
    seen, todo, bad, writes = set(), [(0, False)], set(), 0
    while todo:
        i, pending = todo.pop()
        while i < len(lines) and (i, pending) not in seen:
            seen.add((i, pending))
            ln = lines[i]
            op = ln.split()[0]
            if re.match(r"ds_(write|store)", op):
                pending, writes = True, writes + 1
            elif op == "s_waitcnt" and ("lgkmcnt(0)" in ln or re.fullmatch(r"s_waitcnt\s+0", ln)):
                pending = False
            elif op == "s_barrier" and pending:
                bad.add(i)
            if op == "s_endpgm":
                break
            if op == "s_branch":
                i = label[ln.split()[1]]
                continue
            if op.startswith("s_cbranch"):
                todo.append((label[ln.split()[1]], pending))
            i += 1
    return bad, writes, sum(ln.startswith("s_barrier") for ln in lines)


def test_the_check_sees_a_missing_wait():
    loop = "a:\ns_waitcnt vmcnt(0)\n{}s_barrier\nds_read_b128 v0, v1\nds_write_b128 v1, v[2:5]\ns_cbranch_scc1 a\ns_endpgm\n"
    assert len(_unwaited_barriers(loop.format(""))[0]) == 1
    assert not _unwaited_barriers(loop.format("s_waitcnt lgkmcnt(0)\n"))[0]


@pytest.mark.timeout(600)
def test_lds_writes_are_complete_before_every_barrier(tmp_path):
    src = tmp_path / "k.hip"
    src.write_text('#include "ipc_dma_gemm.h"\nnamespace ipc { namespace dma {\n'
                   + "".join(f"template __global__ void dma_gemm_kernel<{c}>(const Batch);\n" for c in CONFIGS.values())
                   + "} }\n")
    asm = tmp_path / "k.s"
    res = subprocess.run([B.HIPCC, *B.COMMON, "-I", str(B.PKG.parent / "include"), "-I", str(B.CSRC), "--cuda-device-only",
                          "-S", str(src), "-o", str(asm)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    kernels = re.findall(r"^(_Z\w*dma_gemm_kernel\w*):[^\n]*\n(.*?)^\.Lfunc_end\d+:", asm.read_text(), re.S | re.M)
    assert len(kernels) == len(CONFIGS)
    for name, body in kernels:
        bad, writes, barriers = _unwaited_barriers(body)
        assert writes > 0 and barriers >= 2, name
        assert not bad, f"{name}: {len(bad)} of {barriers} barriers with an LDS write in flight"
