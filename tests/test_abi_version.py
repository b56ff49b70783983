"""The library's version number stands for one layout of the header's structures, and the binding has that layout."""
import ctypes
import hashlib
import os
import re
import subprocess

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "pfeife_hip.h")
# version -> digest of the structures: a change of one is a new version, with a line of its own here
LAYOUTS = {5: "18f0ba7bd9fad828", 6: "44ccd84fd201adf4"}


def structures():
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    return {name: " ".join(body.split()) for body, name in re.findall(r"typedef struct \w+ \{(.*?)\} (\w+);", text, flags=re.S)}


def test_a_version_is_one_layout():
    from pfeife_amd import hip

    assert len(structures()) >= 7
    digest = hashlib.sha256(repr(sorted(structures().items())).encode()).hexdigest()[:16]
    assert LAYOUTS.get(hip.load().pf_version()) == digest


def test_the_binding_has_the_headers_layout(tmp_path):
    from pfeife_amd import hip

    pairs = {"pf_gemm_desc": hip.GemmDesc, "pf_job": hip.Job, "pf_norm_bwd_desc": hip.NormBwdDesc, "pf_attn_desc": hip.AttnDesc}
    lines = []
    for name, cls in pairs.items():
        lines.append('printf("%s %%zu\\n", sizeof(%s));' % (name, name))
        for f in cls._fields_:
            lines.append('printf("%s.%s %%zu\\n", offsetof(%s, %s));' % (name, f[0], name, f[0]))
    src = tmp_path / "layout.c"
    src.write_text('#include <stddef.h>\n#include <stdio.h>\n#include "%s"\nint main(void) { %s return 0; }\n' % (HEADER, "\n".join(lines)))
    subprocess.run(["gcc", "-o", str(tmp_path / "layout"), str(src)], check=True)
    got = dict(l.rsplit(" ", 1) for l in subprocess.run([str(tmp_path / "layout")], check=True, capture_output=True, text=True).stdout.splitlines())
    for name, cls in pairs.items():
        assert int(got.pop(name)) == ctypes.sizeof(cls)
        for f in cls._fields_:
            assert int(got.pop("%s.%s" % (name, f[0]))) == getattr(cls, f[0]).offset, f[0]
    assert not got
