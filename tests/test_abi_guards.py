"""The C ABI never throws: every entry point that calls into a device object
(hierarchy, mesh, network), whose members raise on a HIP error, does so inside
a handler. Plain accessors, which touch no device, are listed."""
import pathlib
import re

ABI = pathlib.Path(__file__).resolve().parents[1] / "cfdx_dev_amd" / "csrc" / "abi.cpp"
ACCESSORS = {"num_levels", "level_matrix", "coarse_end_level", "bounded_fallbacks", "n", "reset",
             "npatch", "nc", "nf", "dev", "stream", "h_rowp", "h_cols"}


def _entries(text):
    for m in re.finditer(r"^(?:cfdxhip_status|void|const char\*) (cfdxhip_\w+)\(", text, re.M):
        yield m.group(1), text[m.start():text.index("\n}\n", m.start())]


def test_device_calls_are_guarded():
    entries = list(_entries(ABI.read_text()))
    assert len(entries) > 60
    bare = {}
    for name, body in entries:
        if "guarded(" in body or "try {" in body:
            continue
        calls = set(re.findall(r"(?:dev->|mesh\.|net->|mpnn->)(\w+)", body)) - ACCESSORS
        if calls:
            bare[name] = sorted(calls)
    assert not bare, bare
