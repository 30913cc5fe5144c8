"""bench.py's traffic figures come from committed counter summaries: each says which code it read, and bench.py whether that is the code at
hand (a kernel can be rewritten under its name)."""
import pytest

import bench

PREFILL = {"c1": "gemm_spk_kernel", "c2": "gemm_spk_kernel", "c2_fp32had": "gemm_spk_kernel", "c3": "gemm_sp256_kernel",
           "b13v": "gemm_sp256_kernel", "b70v": "gemm_sp256_kernel", "b13d": "gemm_sp256_kernel", "b70d": "gemm_sp256_kernel"}


@pytest.mark.parametrize("workload", PREFILL)
def test_traffic_of_a_prefill_workload_names_its_code(workload, monkeypatch):
    traffic, source, current = bench.traffic_from_profile(workload, PREFILL[workload])
    assert traffic > 0 and source.startswith("profiles/") and current is not None
    monkeypatch.setattr(bench, "code_digest", lambda source: "0" * 16)
    assert bench.traffic_from_profile(workload, PREFILL[workload]) == (traffic, source, False)


def test_digest_follows_code_and_not_comments(tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    (tmp_path / "quarot_amd" / "csrc").mkdir(parents=True)
    digests = []
    for text in ("int a = 1;\n", "// one\nint  a = 1; /* two\nlines */\n", "int a = 2;\n"):
        (tmp_path / "quarot_amd" / "csrc" / "k.hip").write_text(text)
        digests.append(bench.code_digest("k.hip"))
    assert digests[0] == digests[1] != digests[2]
