"""bench.py divides the counter summaries of `profiles/` by launch times it
measures itself only where the summary was measured on the same kernels (CPU):
comments and spacing may differ, code may not."""

import pytest

import bench

TRAFFIC = "# Traffic\n\nKernel sources: `%s`\n\n| kernel | bytes |\n|---|---|\n| k_vary<true, false> | 1234 | 1 | 1 | 20 |\n"
VALU = ("# Counters\n\nKernel sources: `%s`\n\n## Quintic\n\n| k_vary<true, false> | 20 | 4096 | 77 | 1 | 4.0%% | 60.0%% | 1.90 | 0.006 |\n")


@pytest.mark.parametrize("source,measured", [(None, True), ("0123456789abcdef", False)])
def test_summaries_of_other_kernels_are_not_used(source, measured, tmp_path, monkeypatch):
    for name, text in (("TRAFFIC", TRAFFIC), ("VALU_PROFILE", VALU)):
        path = tmp_path / name
        path.write_text(text % (source or bench.kernel_sources()))
        monkeypatch.setattr(bench, name, str(path))
    assert bench.measured_traffic("k_vary") == (1234.0 if measured else None)
    roof = bench.valu_roofline("k_vary", 0.1, 1e12)
    assert (roof is not None) == measured
    if measured:
        assert roof["achieved"] == pytest.approx(77 * 64 / 1e-4)


def test_comments_are_no_kernels(tmp_path, monkeypatch):
    source = tmp_path / "gagp_amd" / "csrc"
    source.mkdir(parents=True)
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    digests = []
    for text in ("int a = 1;  // one\n", "int a  =  1;\n", "int a = 2;  // one\n"):
        (source / "engine.hip").write_text(text)
        digests.append(bench.kernel_sources())
    assert digests[0] == digests[1] != digests[2]
