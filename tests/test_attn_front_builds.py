"""Which builds of the attention phase can wait for a front of the same launch: only one
that compiles the waits in (MONO_ATTN_FRONT) has done words of a front to name, so a launch
built without them cannot be handed a front whose outputs it would not wait for."""

import subprocess

import pytest

from sgl_amd_mono_amd import build

SOURCE = """
{define}
#include "attn_step.h"
const uint64_t* mono_names_a_front(const mono::attn::Args& a) {{ return a.fdone; }}
"""


def _compiles(tmp_path, define: str) -> tuple[bool, str]:
    src = tmp_path / "names_a_front.hip"
    src.write_text(SOURCE.format(define=define))
    try:
        cc = build.hipcc()
    except RuntimeError as e:
        pytest.skip(str(e))
    res = subprocess.run([cc, *build.COMMON, "-Wno-unused", "--cuda-host-only", "-fsyntax-only", str(src)],
                         capture_output=True, text=True)
    return res.returncode == 0, res.stderr


@pytest.mark.parametrize("define,front", [("#define MONO_ATTN_FRONT 1", True), ("", False),
                                          ("#define MONO_ATTN_LONG 1", False)])
def test_only_a_front_build_names_front_done_words(tmp_path, define, front):
    ok, err = _compiles(tmp_path, define)
    assert ok == front, err
    assert front or "fdone" in err, err
