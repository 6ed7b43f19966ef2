"""CPU: no tuning switch of the kernels decides which memory they touch.

The last lane of a row that its vector does not divide is moved back to end with the row. Whether a
kernel does so must come from the width, as a template parameter of the launch, and never from a
hint mode, which a build may force (-DSIHC_TRI_NTM=3 and the like)."""
from __future__ import annotations

import re
from pathlib import Path

SOURCE = Path(__file__).resolve().parents[1] / "residual-stream-burden_amd" / "csrc" / "sihc_kernels.hip"


def test_ragged_rows_are_not_told_by_a_hint_mode():
    text = SOURCE.read_text()
    derived = re.findall(r"constexpr bool RAG\s*=\s*([^;,]+)[;,]", text)
    assert derived and all(re.fullmatch(r"decltype\(\w+\)::value", d) for d in derived), derived
    kernels = text.split("__global__")
    for before, kernel in zip(kernels, kernels[1:]):
        body = kernel.split("\n}\n", 1)[0]
        if re.search(r"\bRAG\b", body):
            assert "bool RAG" in before[before.rindex("template <"):], kernel[:120]
        for line in body.splitlines():
            if re.search(r"\?[^,;]*lane_channel\(", line):
                assert re.search(r"(RAG|NT) \?", line), line
                if " NT ?" in line:  # whether V divides the width, handed down by the launch as NT
                    assert "bool NT" in before[before.rindex("template <"):], line
