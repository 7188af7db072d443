"""The built kernels' descriptors and places.

No GEMM or combine kernel is launched with scratch: a spilled vector register
adds scratch set-up to every wave of a launch and, in the LDS-ring kernels,
vector-memory operations between copies whose completion is counted by hand
(test_isa_hazards.py, which knows the other vector-memory families).

The decode kernels come before the prefill front end in the engine's code object
(moe_kernels.hip says what their place measured).

Runs on the CPU over the built code object and library; skipped when an artefact
or the ROCm llvm tools are absent."""
import re
import subprocess

import pytest

from test_isa_hazards import ARTEFACTS, LLVM, TARGET

FAMILIES = re.compile(r"netra_moe_(gate_up|down|ffn|combine)_")


def device_object(artefact, tmp_path):
    src = ARTEFACTS[artefact]
    tools = [LLVM / t for t in ("clang-offload-bundler", "llvm-readelf", "llvm-objcopy")]
    if not src.exists() or not all(t.exists() for t in tools):
        pytest.skip("built artefact or ROCm llvm tools not present")
    bundler, readelf, objcopy = map(str, tools)
    bundle, out = src, tmp_path / "gfx950.co"
    if src.suffix == ".so":
        bundle = tmp_path / "fatbin"
        subprocess.run([objcopy, f"--dump-section=.hip_fatbin={bundle}", str(src), str(tmp_path / "so")],
                       check=True, capture_output=True)
    subprocess.run([bundler, "--unbundle", "--type=o", f"--input={bundle}", f"--targets={TARGET}",
                    f"--output={out}"], check=True, capture_output=True)
    return readelf, out


def scratch_bytes(artefact, tmp_path) -> dict[str, int]:
    readelf, out = device_object(artefact, tmp_path)
    notes = subprocess.run([readelf, "--notes", str(out)], check=True, capture_output=True, text=True).stdout
    kernels = notes.split("- .agpr_count")[1:]
    one = lambda k, key: re.search(rf"\.{key}:\s+(\S+)", k).group(1)  # noqa: E731
    return {one(k, "name"): int(one(k, "private_segment_fixed_size")) for k in kernels}


@pytest.mark.parametrize("family", ["gate_up", "down", "ffn", "combine"])
@pytest.mark.parametrize("artefact", sorted(ARTEFACTS))
def test_gemm_kernels_need_no_scratch(artefact, family, tmp_path):
    found = {n: b for n, b in scratch_bytes(artefact, tmp_path).items()
             if (m := FAMILIES.match(n)) and m.group(1) == family}
    assert found or artefact != "hsaco", f"no {family} kernels"
    assert not {n: b for n, b in found.items() if b}


def test_decode_kernels_come_before_the_prefill_front_end(tmp_path):
    readelf, out = device_object("hsaco", tmp_path)
    text = subprocess.run([readelf, "-sW", str(out)], check=True, capture_output=True, text=True).stdout
    at = {f[7]: int(f[1], 16) for f in map(str.split, text.splitlines()) if len(f) > 7 and f[3] == "FUNC"}
    decode = [a for n, a in at.items() if re.match(r"netra_moe_(router_logits|route_h|ffn|gate_up_stream|down_stream|gate_up_split)", n)]
    front = [a for n, a in at.items() if re.match(r"netra_moe_(route_screen|route_select|sort_route)", n)]
    assert decode and front and max(decode) < min(front)
