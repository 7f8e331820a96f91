"""nuc_large_group's narrowing of a tied group, run on the CPU from the kernel's
own source by 512 coroutines with the waves in several orders between barriers
(tests/cpp/narrow_check.cpp): a shared word overwritten before every wave has
read it fails there each time, on a GPU only now and then."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tied_groups_are_narrowed_alike_in_every_wave_order(tmp_path):
    with open(os.path.join(ROOT, "locus_amd", "csrc", "lcs_nucleus.hip")) as f:
        text = f.read()
    start = text.index("struct NucTarget {")
    end = text.index("// The select pass's row finalize:", start)
    assert "nuc_large_group(" in text[start:end]
    (tmp_path / "narrow_group.inc").write_text(text[start:end])
    exe = str(tmp_path / "narrow_check")
    subprocess.run(["g++", "-std=c++20", "-O1", "-w", "-I" + str(tmp_path), "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "narrow_check.cpp")], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout[-4000:])
    assert r.returncode == 0, r.stdout[-4000:]
