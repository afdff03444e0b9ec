"""Which tapes record their forward run (lbm_amd/csrc/record.hpp): a tape whose
fields, mu buffers and gradients fit in free memory is never refused for its
record, whatever the run's length."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
MIB = 1 << 20


def probe(tmp_path, lines):
    exe = tmp_path / "record_probe"
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{ROOT / 'lbm_amd' / 'csrc'}", str(ROOT / "tests" / "record_probe.cpp"),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], input="\n".join(lines) + "\n", check=True, capture_output=True, text=True).stdout
    return [int(v) for v in out.split()]


def granules(n):
    return -(-n // (2 * MIB)) * 2 * MIB


def test_rest_counts_every_buffer(tmp_path):
    # D3Q19 fp32 and fp64 boxes: field, two mu buffers, porosity gradient, wall gradient, target
    for plane, calc, near, target in ((2_200_000, 4, 0, 16384), (17_000_000, 8, 123_456, 65536)):
        field = 19 * plane * calc
        parts = [field, 19 * plane * calc, 19 * plane * calc, 8 * plane, 24 * max(near, 1), 24 * target]
        assert probe(tmp_path, [f"rest {field} {plane} 19 {calc} {near} {target}"]) == [sum(map(granules, parts))]


def test_record_only_beside_everything_else(tmp_path):
    total = 288 << 30
    plane = 100_000_000
    field, step = 76 * plane, 16 * plane
    rest = 3 * granules(field) + granules(8 * plane) + granules(0) + granules(24 * 65536)
    cases = [
        (f"fits 1 {step} {rest} {granules(step) + rest} {total}", 1),       # everything fits exactly
        (f"fits 1 {step} {rest} {granules(step) + rest - 1} {total}", 0),   # a byte short: checkpoints
        (f"fits 1 {step} {rest} {step + 3 * field} {total}", 0),            # room for the fields, not the gradients
        (f"fits 45 {step} {rest} {total} {total}", 1),                      # 72 GB: a quarter of the device
        (f"fits 49 {step} {rest} {total} {total}", 0),                      # more than a quarter
        (f"fits 40 {step} {rest} {80 * step - 1} {total}", 0),              # more than half of what is free
        (f"fits {10 ** 7} {1 << 60} {rest} {total} {total}", 0),            # no overflow
        (f"fits 5 0 {rest} {total} {total}", 0),
    ]
    assert probe(tmp_path, [c for c, _ in cases]) == [v for _, v in cases]
