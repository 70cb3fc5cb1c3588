"""Synchronisation that a run cannot show to be missing: read from the kernels'
sources, since code without it may still come out right as compiled today."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "simd2_amd", "csrc")


def _body(name, function):
    """The braces of `function`, comments taken out."""
    with open(os.path.join(CSRC, name)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    start = text.index("{", re.search(rf"\b{function}\(", text).end())
    depth = 0
    for at in range(start, len(text)):
        depth += {"{": 1, "}": -1}.get(text[at], 0)
        if depth == 0:
            return text[start:at + 1]
    raise AssertionError(f"{function} in {name} does not end")


def test_lds_exchange_of_the_wave_kernel_is_fenced():
    """Lanes of a wave read what other lanes stored, with no barrier: between the
    stores and the reads on either side of them stands a wave fence."""
    loop = _body("srgemm_valu.hip", "wave_loop")
    stores = list(re.finditer(r"(?<!auto )\bstore\([^)]*\);", loop))
    assert len(stores) == 2  # the first slab's and the loop's
    for m in stores:
        assert re.match(r"\s*wave_lds_fence\(\);", loop[m.end():])
    assert re.search(r"wave_lds_fence\(\);\s*$", loop[:stores[1].start()])
    # the partial tile is parked over slabs that other lanes have read
    kernel = _body("srgemm_valu.hip", "srgemm_wave_kernel")
    assert re.search(r"wave_loop<Op>\([^;]*;.*?wave_lds_fence\(\);.*?\bpart\[", kernel, re.S)


def test_symmetry_check_leaves_as_one_workgroup():
    """Other workgroups write *asym during the launch, so waves may read different
    values: the decision to leave is taken by the workgroup, after a barrier."""
    body = _body("sched.hip", "symmetry_check_kernel")
    before = body[:body.index("return;")]
    assert "__syncthreads" in before and "__hip_atomic_load(asym" in before
    assert not re.search(r"\*asym\b(?! = 1;)", body)
