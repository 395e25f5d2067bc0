"""The HBM traffic that the bench quotes is of the kernel that it times: a recorded run of another
kernel of the same precision and walker count is not taken."""
import bench


def test_traffic_of_another_kernel_is_not_quoted(tmp_path, monkeypatch):
    (tmp_path / "profiles").mkdir()
    rows = ["# kernel\tprecision\twalkers\tread\twrite\tsource",
            "k_sweep_mx<64,1,0,8,1> (32 moves per launch)\tmixed_fp32\t8192\t629695216\t501079520\told.md"]
    (tmp_path / "profiles" / "traffic.tsv").write_text("\n".join(rows) + "\n")
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.profile_traffic("mixed_fp32", 8192) is None
    rows.append("k_sweep_mxp<64,1,true,false> (32 moves per launch)\tmixed_fp32\t8192\t5\t7\tnew.md")
    (tmp_path / "profiles" / "traffic.tsv").write_text("\n".join(rows) + "\n")
    assert bench.profile_traffic("mixed_fp32", 8192) == 12
    assert bench.profile_traffic("fp64", 8192) is None and bench.profile_traffic("mixed_fp32", 4096) is None
