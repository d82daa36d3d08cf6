"""Every entry point that works on the device selects its context's (or plan's) device first: a
host thread may hold contexts of several devices, and a block allocated on the wrong one would
stay in the context's pool.  Read from the source: one device is all a test machine has."""
import pathlib
import re

SRC = pathlib.Path(__file__).resolve().parents[1] / "boundaryvaluediffeq.jl_amd" / "csrc" / "bvp_api.hip"

# no device memory, stream or event is touched
HOST_ONLY = {"bvp_opts_default", "bvp_last_error", "bvp_batch_info", "bvp_batch_chunking", "bvp_batch_set_chunking",
             "bvp_batch_precision", "bvp_batch_set_config", "bvp_batch_config", "bvp_batch_timing",
             "bvp_batch_set_graph", "bvp_mlp_set_normalization"}
# only pass their arguments on to a function that selects it
FORWARD = {"bvp_firk_residual", "bvp_firk_newton_step", "bvp_firk_defect"}


def _entries():
    text = SRC.read_text()
    text = text[text.index('extern "C" {'):]
    return re.findall(r"^(?:int|void|const char \*) ?(bvp_\w+)\([^)]*\) (\{.*?^\}|\{.*?\}$)", text, re.M | re.S)


def test_every_entry_point_selects_its_device():
    found = dict(_entries())
    assert len(found) >= 40 and HOST_ONLY | FORWARD <= set(found)
    for name, body in found.items():
        if name in HOST_ONLY:
            continue
        if name in FORWARD:
            assert "firk_component(ctx," in body
            continue
        sel = body.find("hipSetDevice(")
        assert sel >= 0, name
        work = [body.find(w) for w in ("hipMemcpy", "hipEvent", "hipStream", "dalloc(", "run_component(", "batch_build(",
                                       "batch_run(", "batch_sync(", "batch_results(", "enqueue_", "delete ")]
        assert all(w < 0 or w > sel for w in work), name


def test_the_forwarded_call_selects_it():
    text = SRC.read_text()
    body = text[text.index("static int firk_component("):]
    assert "hipSetDevice(ctx->device)" in body[:body.index("\n}\n")]
