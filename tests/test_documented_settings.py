"""Every setting that docs/ENVIRONMENT.md names is read somewhere: a setting whose reader went away would be accepted and do
nothing."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_documented_settings_are_read():
    path = os.path.join(ROOT, "docs", "ENVIRONMENT.md")
    with open(path) as f:
        names = set(re.findall(r"`(MXS_[A-Z0-9_]+)`", f.read()))
    assert {"MXS_SAMPLE_REG", "MXS_MPLAN", "MXS_GEMM_PF"} <= names
    text = ""
    for pattern in ("*.py", "*.sh", "mxserve/**/*.py", "csrc/**/*", "scripts/**/*", "deploy/**/*"):
        for fn in glob.glob(os.path.join(ROOT, pattern), recursive=True):
            if os.path.isfile(fn):
                with open(fn, errors="replace") as f:
                    text += f.read()
    unread = sorted(n for n in names if not re.search(re.escape(n) + r"\b", text))
    assert not unread, unread
