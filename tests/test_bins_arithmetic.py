"""Entries per work item of the binned deposit at the largest bunches: a mesh of
one brick (or a dense core) puts up to 2^32 - 1 particles into one brick.  The
device function is constexpr and evaluated by the compiler on the host, so no
bunch of that size is needed."""
import os
import subprocess

import pytest

from ocelot_amd import build

CSRC = os.path.join(build.HERE, "csrc")


def _holds(tmp_path, asserts):
    src = tmp_path / "t.hip"
    src.write_text('#include "bins.hpp"\nusing namespace ocsc;\n' + "".join(f"static_assert({a});\n" for a in asserts))
    r = subprocess.run([build.hipcc(), "--offload-host-only", "-std=c++17", "-fsyntax-only", "-I", CSRC, str(src)],
                       capture_output=True, text=True)
    return r.returncode == 0, r.stderr[-2000:]


@pytest.mark.parametrize("total", [1, 8191, 8192, 8193, 2 ** 31 - 1, 2 ** 31, 2 ** 31 + 1, 2 ** 32 - 1])
def test_chunks_cover_a_brick(tmp_path, total):
    chunk = 8192
    items = -(-total // chunk)
    at = sorted({0, 1, items // 3, items // 2, items - 2, items - 1} & set(range(items)))
    ok, err = _holds(tmp_path, ["kBinChunk == 8192"] + [
        f"bin_chunk_entries({total}u, {k}) == {min(chunk, total - k * chunk)}" for k in at])
    assert ok, err
