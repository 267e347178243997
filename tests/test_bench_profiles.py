"""The counter summaries that bench.py divides by live launch times belong to the kernels as they are built."""
import json

import pytest

import bench

KERNELS = ["Q8_0", "Q4_0", "Q2K", "Q3K", "Q4K", "Q5K", "Q6K", "IQ4_XS", "IQ3_XXS", "IQ2_XS", "IQ1_S", "IQ1_M"]


@pytest.mark.parametrize("kernel", KERNELS)
def test_counts_are_used_for_their_own_source_only(kernel, tmp_path, monkeypatch):
    """a count taken on another source gives None; edits of comments and layout change nothing"""
    csrc = tmp_path / "seedpack_amd" / "csrc"
    csrc.mkdir(parents=True)
    (tmp_path / "profiles").mkdir()
    for p in bench._kernel_sources(kernel):
        (csrc / p.rsplit("/", 1)[1]).write_text(open(p).read())
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    d = {"sources": {kernel: bench.source_digest(kernel)}, "insts_valu_per_launch": {kernel: 1000},
         "bytes_per_launch": {kernel: 77}, "issue": {kernel: {"issue_slot_occupancy": 0.5}}}
    for name in ("valu.json", "traffic.json"):
        (tmp_path / "profiles" / name).write_text(json.dumps(d))
    figures = lambda: (bench._profiled_valu(kernel), bench._profiled_issue(kernel), bench._profiled_traffic(kernel))
    assert figures() == (64000, 0.5, 77)
    own = bench._kernel_sources(kernel)[0]
    text = open(own).read()
    open(own, "w").write("// a note\n/* another\n one */" + text.replace("    ", "  "))
    assert figures() == (64000, 0.5, 77)
    open(own, "w").write(text.replace("constexpr", "static constexpr", 1))
    assert figures() == (None, None, None)
    open(own, "w").write(text)
    shared = bench._kernel_sources(kernel)[1]
    open(shared, "a").write("int added;\n")
    assert figures() == (None, None, None)


def test_the_committed_summaries_name_their_sources():
    for name, section in (("valu.json", "insts_valu_per_launch"), ("traffic.json", "bytes_per_launch")):
        d = json.load(open(f"{bench.ROOT}/profiles/{name}"))
        assert set(d[section]) <= set(d["sources"]), name
