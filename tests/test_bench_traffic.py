"""bench.py's traffic figures come from committed counter summaries: each says which code it read, and bench.py whether that is the code at
hand (a kernel can be rewritten under its name)."""
import pytest

import bench

PREFILL = ("c1", "c2", "c2_fp32had", "c3", "b13v", "b70v", "b13d", "b70d")


def _launched(workload):
    m, k, n = bench.WORKLOADS[workload][:3] if bench.WORKLOADS[workload] else (32768, 4096, 12288)
    return bench.gemm_kernel_name(m, n, k)


@pytest.mark.parametrize("workload", PREFILL)
def test_traffic_of_a_prefill_workload_names_its_code(workload, monkeypatch):
    """For the kernels that bench.py reports: what the library launches with the scratch that the package gives it."""
    kernel = _launched(workload)
    traffic, source, current = bench.traffic_from_profile(workload, kernel)
    assert traffic > 0 and source.startswith("profiles/") and current is not None
    monkeypatch.setattr(bench, "code_digest", lambda source: "0" * 16)
    assert bench.traffic_from_profile(workload, kernel) == (traffic, source, False)


@pytest.mark.parametrize("workload", ("c3", "b13d", "b70d"))
def test_traffic_of_two_launches_is_their_sum_and_of_their_code(workload, monkeypatch):
    """A summary that holds readings of the kernel that runs without scratch and of the two that run with it."""
    kernel = _launched(workload)
    assert kernel.startswith("spread_x6_kernel + gemm_x6_kernel")
    of = lambda kernel: bench.traffic_from_profile(workload, kernel)[0]
    assert abs(of(kernel) - of("spread_x6_kernel") - of("gemm_x6_kernel")) <= 2 and of("spread_x6_kernel") > 0      # (each rounded)
    assert of("gemm_sp256_kernel") > 0 and of("gemm_sp256_kernel") != of("gemm_x6_kernel")
    asked = []
    monkeypatch.setattr(bench, "code_digest", lambda source: asked.append(source))
    for name in (kernel, "gemm_sp256_kernel"):
        bench.traffic_from_profile(workload, name)
    assert asked == ["gemm_x6.hip", "gemm_e2m3.hip"]


def test_digest_follows_code_and_not_comments(tmp_path, monkeypatch):
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    (tmp_path / "quarot_amd" / "csrc").mkdir(parents=True)
    digests = []
    for text in ("int a = 1;\n", "// one\nint  a = 1; /* two\nlines */\n", "int a = 2;\n"):
        (tmp_path / "quarot_amd" / "csrc" / "k.hip").write_text(text)
        digests.append(bench.code_digest("k.hip"))
    assert digests[0] == digests[1] != digests[2]
