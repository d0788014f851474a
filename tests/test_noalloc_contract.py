"""hipclaw_step_batch_noalloc allocates nothing (include/hipclaw.h): neither its body
nor the scratch lookup it calls names an allocation, on the device or on the host."""
import os
import re

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "forestclaw_amd", "csrc", "hipclaw_capi.hip")


def _body(text, head):
    i = text.index("{", text.index(head))
    depth, j = 0, i
    while True:
        depth += {"{": 1, "}": -1}.get(text[j], 0)
        j += 1
        if depth == 0:
            return re.sub(r"//[^\n]*", "", text[i:j])


def test_no_allocation_is_named():
    with open(SRC) as f:
        text = f.read()
    for head in ("int hipclaw_step_batch_noalloc(", "static void* scratch_ptr("):
        body = _body(text, head)
        found = re.findall(r"\bnew\b|\w*[mM]alloc\w*|\w*calloc\w*|unique_ptr|make_\w+|std::vector|std::string|resize|push_back", body)
        assert not found, (head, found)
