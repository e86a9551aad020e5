"""Host-side checks of bench.py (no GPU): the one-GPU contract of the
command line and the CPU leg's per-config table."""
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def test_bench_refuses_more_than_one_gpu():
    """``--gpus N`` with N > 1 exits with status 2 and says why (every box
    here has one GPU; the sharding is design only), before touching a GPU."""
    res = subprocess.run([sys.executable, str(ROOT / "bench.py"), "--gpus", "2"], cwd=ROOT,
                         capture_output=True, text=True, timeout=300)
    assert res.returncode == 2
    assert "one GPU" in res.stderr or "1 GPU" in res.stderr or "--gpus 1" in res.stderr


def test_cpu_kernel_table_on_host():
    """The CPU leg times configs 1-4 through the oracle ops on the host: every
    config of the GPU table has a positive time and a byte rate."""
    sys.path.insert(0, str(ROOT))
    import torch

    import bench

    torch.set_num_threads(min(8, torch.get_num_threads()))
    out = bench.cpu_kernel_table()
    names = {"cfg1_resnorm_gemv_6144x2048", "cfg3_gqa_decode_L512", "cfg3_gqa_decode_L8192",
             "cfg4_delta_decode_chain_per_token"}
    names |= {f"cfg2_a8w8_{s}_m{m}" for s in ("12288x2048", "2048x6144") for m in (1, 4, 16)}
    assert names <= set(out)
    for rec in out.values():
        assert rec["us"] > 0 and rec["GB/s"] > 0


RING = "void (anonymous namespace)::gemm_ring<2, 2, 2, 1, 128, 6, 8, true, {}, false, false>(GemmArgs)"
KSPLIT = "void (anonymous namespace)::gemm_ksplit<2, 2, 4, 2, false, {}>(GemmArgs)"


def _trace(path, names):
    rows = ["Dispatch_Id,Kernel_Name,Grid_Size_X,Start_Timestamp,End_Timestamp"]
    rows += [f'{i},"{n}",256,{10000 * i},{10000 * i + 5000}' for i, n in enumerate(names)]
    path.write_text("\n".join(rows))
    return str(path)


def test_vision_trace_of_the_own_gemms(tmp_path, capsys):
    """The tower's table runs from the patch embedding to the merger's copies
    whichever kernel its last product is on."""
    import bench

    tower = [KSPLIT.format(5), "position_embed_add_rows<true>()", RING.format(5), RING.format(6)]
    ours = tower + [KSPLIT.format(5), "__amd_rocclr_copyBuffer", "__amd_rocclr_copyBuffer"]
    library = tower + ["Cijk_Alik", "__amd_rocclr_copyBuffer", "__amd_rocclr_copyBuffer"]
    (tmp_path / "b.json").write_text('{"vision_tower": {}}')
    for call in (ours, library):
        trace = _trace(tmp_path / "t.csv", ["Cijk_Alik"] * 9 + call + ["top1"])
        bench.trace_summary("vision", trace, str(tmp_path / "b.json"))
        assert "7 kernels" in capsys.readouterr().out


def test_matrix_core_table_counts_every_gemm(tmp_path, capsys):
    """The probe's products are labelled in order, those on the K-splitting
    kernel among them."""
    import bench

    names = [(KSPLIT if n == 2048 else RING).format(3 if int8 else 0)
             for n, _, _ in bench.PROBE_GEMMS for int8 in (False, True) for _ in range(3)]
    trace = _trace(tmp_path / "t.csv", [RING.format(0)] * 5 + names)
    rows = ["Dispatch_Id,Kernel_Name,Counter_Name,Counter_Value"]
    rows += [f'{i},"{n}",SQ_INSTS_VALU_MFMA_MOPS_{"I8" if ", 3" in n else "BF16"},1e9'
             for i, n in enumerate([RING.format(0)] * 5 + names)]
    (tmp_path / "c.csv").write_text("\n".join(rows))
    bench.mfma_summary(str(tmp_path / "c.csv"), trace)
    table = capsys.readouterr().out.splitlines()[1:]
    assert len(table) == 2 * len(bench.PROBE_GEMMS)
    assert all(("gemm_ksplit" in row) == row.startswith("2048x") for row in table)
    assert all(" | 0.0000 | " not in row for row in table)
