"""Scratch slots are process-wide buffers: a slot that two source files name would be shared by
entry points that may run at the same time on different threads and streams."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "yasps_amd" / "csrc"
# run-time parts of a slot number and the values they take
RANGES = {"tree": range(2), "t": range(5), "s": [80, 96], "slot_base": [15, 20]}


def _slots(text):
    found = set()
    for expr in re.findall(r"\bscratch\(\s*([^,()]+),\s*[^)]", text):
        if expr.startswith("int "):
            continue                                     # its declaration and definition
        names = [n for n in RANGES if re.search(rf"\b{n}\b", expr)]
        assert len(names) <= 1, expr
        values = [{names[0]: v} for v in RANGES[names[0]]] if names else [{}]
        found |= {eval(expr, {"__builtins__": {}}, v) for v in values}
    return found


def test_every_slot_belongs_to_one_file():
    files = {p.name: _slots(p.read_text()) for p in sorted(CSRC.iterdir())
             if p.suffix in (".hip", ".hpp")}
    assert {len(files[n]) > 0 for n in ("tiles.hip", "jacobian.hip", "ccd.hip", "indices.hip",
                                        "bsr3.hip", "energy_kernels.hpp")} == {True}
    owner = {}
    for name, slots in files.items():
        for slot in slots:
            assert owner.setdefault(slot, name) == name, f"slot {slot}: {owner[slot]} and {name}"
