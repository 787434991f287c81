"""The arrival counters of the one-launch reductions: whatever clears one of them clears all (a stale one lets a block finish a
tile whose other parts have not arrived)."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "seq2seqsharp_amd", "csrc")


def test_counters_are_cleared_together():
    text = open(os.path.join(CSRC, "tship_gpt.hip")).read()
    model = text[text.index("struct TSHipGpt {"):text.index("\n};", text.index("struct TSHipGpt {"))]
    names = {n for line in re.findall(r"DevBuf ([^;(){}]+);", model) for n in re.split(r",\s*", line) if n.endswith("_count")}
    assert names >= {"tile_count", "attn_count", "mid_count"}
    body = re.search(r"void clear_counters\(\) \{.*?\n    \}", model, re.S).group(0)
    assert all("&" + n in body for n in names), names
    for entry in ("TSHip_GptReset(TSHipGpt* m)", "static int generate_impl("):
        at = text.index(entry)
        assert "clear_counters()" in text[at:text.index("\n}\n", at)], entry
    # nothing clears one of them by itself behind its allocation (which is of no concern to a later step)
    assert not re.findall(r"hipMemsetAsync\(m->\w+_count", text)
