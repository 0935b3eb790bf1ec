"""CPU tests on the compiler's listing of the workspace route's product kernel (csrc/kernels/gram_f16_wide.hpp).

The kernel's operands, and behind the walk the staging of its results, share one array in LDS, which the waves of a workgroup fill
and read in turn.  A wave that stages over what another has yet to read gives wrong numbers only when the two happen to be
far enough apart, which no run of the kernel shows reliably.  The order is therefore checked where it is certain: over every path through
the compiled kernel.
"""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from kermac_amd import _build

KERNELS = Path(_build.CSRC) / "kernels"
VARIANTS = [(tile, symmetric, epilogue) for tile in ("WideTileLarge", "WideTileSmall")
            for symmetric, epilogue in (("true", "GW_EPILOGUE_DISTANCE"), ("false", "GW_EPILOGUE_DISTANCE"),
                                        ("true", "GW_EPILOGUE_DOT"), ("false", "GW_EPILOGUE_GRADIENT_L2"))]


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    if shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists():
        pytest.skip("no hipcc")
    folder = tmp_path_factory.mktemp("listing")
    source, target = folder / "product.hip", folder / "product.s"
    source.write_text("#include <hip/hip_runtime.h>\n" f'#include "{KERNELS / "gram_f16_wide.hpp"}"\n'
                      + "".join(f"template __global__ void kmc::gram_f16_wide<kmc::{tile}, {symmetric}, kmc::{epilogue}>(kmc::GramWideArgs);\n"
                                for tile, symmetric, epilogue in VARIANTS))
    done = subprocess.run([_build._hipcc(), *_build.HIPCC_FLAGS, "--offload-device-only", "-S", str(source), "-o", str(target)],
                          capture_output=True, text=True)
    assert done.returncode == 0, done.stderr[-2000:]
    return functions(target.read_text())


def functions(text):
    """name -> list of (label or None, instruction text), one entry per line that is either."""
    found, lines = {}, None
    for line in text.splitlines():
        start = re.match(r"(_Z\w*gram_f16_wide\w*):", line)
        if start:
            lines = found.setdefault(start.group(1), [])
        elif lines is not None:
            if line.startswith(".Lfunc_end"):
                lines = None
                continue
            label = re.match(r"(\.LBB\w+):", line)
            body = line.split(";")[0].strip() or ("wave_barrier" if "; wave barrier" in line else "")
            if label:
                lines.append((label.group(1), ""))
            elif body and not body.startswith("."):
                lines.append((None, body))
    return found


def successors(lines):
    at_label = {label: at for at, (label, _) in enumerate(lines) if label}
    follow = []
    for at, (_, body) in enumerate(lines):
        op = body.split()[0] if body else ""
        assert not op.startswith(("s_setpc", "s_swappc", "s_call")), body
        if op == "s_endpgm":
            follow.append([])
        elif op == "s_branch":
            follow.append([at_label[body.split()[1]]])
        elif op.startswith("s_cbranch"):
            follow.append([at_label[body.split()[1]], at + 1])
        else:
            follow.append([at + 1] if at + 1 < len(lines) else [])
    return follow


def reachable(starts, follow, stop=lambda at: False):
    """Everything that an execution can come to behind `starts`, not going on behind what `stop` names."""
    seen, todo = set(), [s for at in starts for s in follow[at]]
    while todo:
        at = todo.pop()
        if at in seen:
            continue
        seen.add(at)
        if not stop(at):
            todo += follow[at]
    return seen


class Listing:
    def __init__(self, lines):
        self.lines, self.follow = lines, successors(lines)
        self.ops = [body.split()[0] if body else "" for _, body in lines]
        self.products = [at for at, op in enumerate(self.ops) if op.startswith("v_mfma")]
        behind = [[] for _ in lines]
        for at, after in enumerate(self.follow):
            for s in after:
                behind[s].append(at)
        self.before_a_product = reachable(self.products, behind)
        self.after_a_product = reachable(self.products, self.follow)

    def all(self, *prefixes):
        return [at for at, op in enumerate(self.ops) if op.startswith(prefixes)]


def test_every_variant_is_listed(listings):
    assert len(listings) == len(VARIANTS)
    assert all(len(Listing(lines).products) >= 48 for lines in listings.values())


def test_no_wave_stages_results_over_operands_that_another_has_yet_to_read(listings):
    """Between any read of operands and any write to LDS behind the walk there is a barrier, on every path."""
    for name, lines in listings.items():
        code = Listing(lines)
        reads = [at for at in code.all("ds_read", "ds_load") if at in code.before_a_product]
        staged = {at for at in code.all("ds_write", "ds_store") if at not in code.before_a_product}
        assert reads
        without = reachable(reads, code.follow, stop=lambda at: code.ops[at] == "s_barrier") & staged
        assert not without, f"{name}: {[lines[at][1] for at in sorted(without)][:4]}"


def test_lanes_of_a_wave_exchange_staged_results_in_order(listings):
    """Lanes of a wave hand results to each other through LDS.  The compiler has to respect the order within one lane only, so a
    barrier of the wave keeps the reads behind the other lanes' writes, and the next writes behind those reads."""
    for name, lines in listings.items():
        code = Listing(lines)
        barrier = lambda at: code.ops[at] == "s_barrier"
        ordered = lambda at: code.ops[at] in ("s_barrier", "wave_barrier")
        reads = {at for at in code.all("ds_read", "ds_load") if at not in code.before_a_product}
        # what is written and read with no barrier of the workgroup in between is exchanged within a wave
        exchanged = {at for at in code.all("ds_write", "ds_store") if at not in code.before_a_product
                     and reachable([at], code.follow, stop=barrier) & reads}
        assert bool(exchanged) == ("ELi1EEEv" not in name), name        # the gradient's epilogue (1) stages nothing
        early = reachable(exchanged, code.follow, stop=ordered) & reads
        assert not early, name
        behind = reads & reachable(exchanged, code.follow, stop=barrier)
        overwritten = reachable(behind, code.follow, stop=ordered) & exchanged
        assert not overwritten, name


def registers(text):
    found = set()
    for first, last in re.findall(r"\bv\[(\d+):(\d+)\]", text):
        found |= set(range(int(first), int(last) + 1))
    return found | {int(at) for at in re.findall(r"\bv(\d+)\b", text)}


def test_nothing_but_the_products_touches_the_sums_in_the_walk(listings):
    """The matrix instructions are inline assembly, so the compiler keeps no distance between one of them and an instruction that reads or
    moves its sums.  Inside the walk there must be no such instruction; behind it only past the wait states that end it."""
    for name, lines in listings.items():
        code = Listing(lines)
        products = set(code.products)
        sums = set().union(*(registers(lines[at][1].split(",")[0]) for at in products))
        for at in products:
            to, _, _, added = (registers(x) for x in re.findall(r"v\[\d+:\d+\]", lines[at][1]))
            assert to == added, "the sums stay in their registers"
        # the wait states: at least 16 behind the last product before anything else reads or writes a sum
        waited = lambda at: lines[at][1] == "s_nop 15"
        close = reachable(products, code.follow, stop=waited) - products
        for at in sorted(close):
            assert not registers(lines[at][1]) & sums, f"{name}: {lines[at][1]}"
        assert not code.all("scratch_", "buffer_store", "buffer_load"), f"{name} spills"
