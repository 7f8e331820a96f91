"""The lm-head's choice of a tile (lmhead_shape, lcs_lmhead.hip), compiled for the
CPU from the kernel's source: the GPU tests' list of steady-state cases names
the tile that each runs on, and every tile has one."""
import ctypes
import os
import re
import subprocess

from tests.test_gpu_lmhead import STEADY

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CUS = 256


def test_steady_cases_cover_every_tile(tmp_path):
    with open(os.path.join(ROOT, "locus_amd", "csrc", "lcs_lmhead.hip")) as f:
        text = f.read()
    rule = text[text.index("struct LmShape {"):text.index("hipError_t launch_lmhead(")]
    with open(os.path.join(ROOT, "locus_amd", "csrc", "lcs_internal.hpp")) as f:
        consts = re.findall(r"^constexpr uint32_t (?:kMaxVocab|kLmMaxBlocks) = .*$", f.read(), re.M)
    assert len(consts) == 2
    big = re.search(r"^constexpr uint32_t kBigHidden = .*$", text, re.M).group(0)
    (tmp_path / "shape.cpp").write_text(
        "#include <cstdint>\n" + "\n".join(consts) + "\n" + big + "\n" + rule +
        """extern "C" void shape(uint32_t rows, uint32_t vocab, uint32_t hidden, uint32_t cus, uint32_t* o) {
    const LmShape s = lmhead_shape(rows, vocab, hidden, cus);
    o[0] = s.vt, o[1] = s.br;
}
""")
    so = str(tmp_path / "shape.so")
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-o", so, str(tmp_path / "shape.cpp")], check=True, timeout=120)
    fn = ctypes.CDLL(so).shape
    out = (ctypes.c_uint32 * 2)()
    seen = set()
    for rows, vocab, vt, br, ks, st in STEADY:
        fn(rows, vocab, 320, CUS, out)
        assert tuple(out) == (vt, br), (rows, vocab, tuple(out))
        blocks = -(-vocab // (64 * vt))
        # launch_lmhead's forms: 64-k stages for two 256-column tiles a CU and the 256 x 256 tile
        wide = (vt, br) == (4, 256) or ((vt, br) == (4, 64) and CUS < blocks <= 2 * CUS)
        assert (ks == 4) == wide, (rows, vocab)
        assert 320 // (16 * ks) > st, (rows, vocab)   # more stages than the ring holds
        seen.add((vt, br, ks, st, rows > br))
    launched = set()
    for m in re.findall(r"\(lmhead_tile<([^>]*)>\)", text):
        a = [x.strip() for x in m.split(",")]
        if len(a) < 6:   # (the last argument: row offsets past 32 bits, tested apart)
            launched.add((int(a[0]), int(a[1]), int(a[4]) if len(a) > 4 else 2, int(a[2])))
    assert launched == {s[:4] for s in seen}, launched ^ {s[:4] for s in seen}
    # tiles of 128 and 256 rows, also with several row tiles
    assert {s[:2] for s in seen if s[4]} >= {(2, 128), (4, 128), (2, 256), (4, 256)}
