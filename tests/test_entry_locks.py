"""The C entry points' thread safety, read from the source: an entry point that
touches what calls on one context share (its buffers, its pending scratch, its
launch table) holds the context's mutex from before the first touch."""
import re
from pathlib import Path

SRC = Path(__file__).resolve().parents[1] / "film_grain_amd" / "csrc" / "fg_capi.hip"

# set at creation and never changed, atomic, or per call (the error text)
OWN = {"device", "max_lds", "num_cus", "mu", "last_error", "noalloc_scratch", "h_cancel", "d_cancel"}
# helpers that take the context and touch none of what calls share, and those
# that take the mutex themselves
FREE = {"set_error", "hip_error", "validate", "validate_frame", "set_cancel", "render_host", "stats_device"}
# creation and destruction, and the error text's reader
EXEMPT = {"fg_ctx_create", "fg_ctx_destroy", "fg_last_error"}


def _code():
    text = SRC.read_text()
    text = re.sub(r"/\*.*?\*/", " ", text, flags=re.S)
    return re.sub(r"//[^\n]*", " ", text)


def _body(code, at):
    start = code.index("{", at)
    depth, i = 0, start
    while True:
        depth += {"{": 1, "}": -1}.get(code[i], 0)
        i += 1
        if depth == 0:
            return code[start:i]


def _members(code):
    body = _body(code, code.index("struct fg_ctx {"))
    names = set()
    for decl in re.sub(r"\{[^{}]*\}", "", body[1:-1]).split(";"):
        decl = re.sub(r"<[^<>]*(<[^<>]*>)?[^<>]*>", "", decl)
        decl = re.sub(r"\[[^\]]*\]|=[^,]*", "", decl)
        if decl.strip():
            names.update(re.sub(r".*[\s*]", "", part.strip(), flags=re.S) for part in decl.split(","))
    return names


def _first_touch(body, members):
    found = [m.start() for m in re.finditer(r"\bctx->(\w+)", body) if m.group(1) in members - OWN]
    found += [m.start() for m in re.finditer(r"\b(\w+)\((?:b->)?ctx\s*[,)]", body) if m.group(1) not in FREE | {"lock"}]
    return min(found, default=None)


def test_entry_points_hold_the_mutex():
    code = _code()
    members = _members(code)
    assert {"stream", "scratch_pending", "cells", "scale_state", "table", "pub_seq", "tev"} <= members
    entries = [(m.group(1), m.start()) for m in
               re.finditer(r"^(?:int|void|const char \*)\s*(fg_\w+)\((?:const )?fg_(?:ctx|batch) \*[^;{]*\{", code, re.M)]
    assert len(entries) > 35
    touching = []
    for name, at in entries:
        if name in EXEMPT:
            continue
        body = _body(code, at)
        touch = _first_touch(body, members)
        if touch is None:
            continue
        touching.append(name)
        lock = re.search(r"lock_guard<std::mutex> lock\((?:b->)?ctx->mu\)", body)
        assert lock and lock.start() < touch, name
    assert {"fg_budget_scale_device", "fg_lambda_device", "fg_render_frame_device"} <= set(touching)
