"""What the GEMM kernels may read of a strided operand or scale matrix (CPU only):
rows_bytes and rows_bytes_f32, the extent of a buffer descriptor, against the
bytes that the rows use, and every kernel's descriptors, which must be built with
them."""
import glob
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gcnasm_amd",
                    "csrc")

CHECK = r"""
#include "ga_extent.hpp"
#include <stdio.h>
int main()
{
    int bad = 0;
    // the last row's last used byte is the last one covered
    const long long rows_of[] = {1, 2, 17, 64, 128, 8192}, used_of[] = {128, 512, 7168};
    const long long pad_of[] = {0, 16, 128, 4096};
    for (long long rows : rows_of)
        for (long long used : used_of)
            for (long long pad : pad_of) {
                const long long ld = used + pad, storage = (rows - 1) * ld + used;
                bad += (long long)ga::rows_bytes(rows, ld, used) != storage;
                bad += (long long)ga::rows_bytes_f32(rows, ld / 4, used / 4) != storage;
            }
    // at most 4 GiB less 16 bytes
    bad += ga::rows_bytes(256, 1ll << 26, 1ll << 26) != 0xFFFFFFF0u;
    bad += ga::rows_bytes(255, 16842752, 4096) != 254u * 16842752u + 4096u;
    printf("%d\n", bad);
    return 0;
}
"""


def test_rows_bytes(tmp_path):
    src = tmp_path / "extent.cpp"
    src.write_text(CHECK)
    exe = str(tmp_path / "extent")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, "-o", exe, str(src)], check=True)
    assert subprocess.run([exe], check=True, capture_output=True, text=True).stdout.strip() == "0"


def descriptors(path):
    """The size argument of every make_rsrc call."""
    text = re.sub(r"//.*", "", open(path).read())
    out = []
    for m in re.finditer(r"\bmake_rsrc\(", text):
        depth, i, args, start = 1, m.end(), [], m.end()
        while depth:
            c = text[i]
            depth += (c in "([{") - (c in ")]}")
            if (c == "," and depth == 1) or depth == 0:
                args.append(" ".join(text[start:i].split()))
                start = i + 1
            i += 1
        out.append(args)
    return out


# Sizes that are no strided rows: MX scales (padded and shuffled, a dense matrix),
# preshuffled B (16-row groups of K * 16 contiguous bytes) and stream-K's slots.
DENSE = [r"\(uint32_t\)\(+(\(int\)args\.)?M \+ 31\) / 32 \* 32\) \* sna", r"\(uint32_t\)sma \* sna",
         r"\(uint32_t\)\(+N \+ 31\) / 32 \* 32\) \* snb", r"\(uint32_t\)smb \* snb",
         r"\(uint32_t\)(ng_here|ngb) \* \(uint32_t\)Kb \* 16", r"kSkSlotFloats \* 4"]
SOURCES = sorted(glob.glob(os.path.join(CSRC, "gemm_[bm]*.hip")))


@pytest.mark.parametrize("path", SOURCES, ids=[os.path.basename(p) for p in SOURCES])
def test_descriptors_end_with_the_rows(path):
    found = descriptors(path)
    assert all(len(a) == 2 for a in found)
    for _, size in found:
        assert re.match(r"(ngb > 0 \? )?rows_bytes(_f32)?\(", size) or any(
            re.fullmatch(d, size) for d in DENSE), size
    assert found
