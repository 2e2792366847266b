"""CPU check that the recorded HBM traffic bench.py attaches to its entries
names kernels that the sources still hold."""
import json
import re
from pathlib import Path

REPO = Path(__file__).resolve().parents[1]


def test_traffic_kernels_exist():
    src = "".join(p.read_text() for p in (REPO / "ternary-bonsai-inference_amd" / "csrc").glob("*.hip"))
    data = json.loads((REPO / "profiles" / "traffic_all_configs.json").read_text())
    names = {re.match(r"\w+", k).group() for e in data["entries"] for k in e["kernels"]}
    missing = sorted(n for n in names if not re.search(rf"\b{n}\(", src))
    assert not missing, missing
