"""The build's reading of the compiler's resource report: a path kernel whose
vector registers went to memory does not pass."""
import pytest

from prender_amd import build as B


def report(kernels):
    lines = []
    for name, vgprs, sspill, vspill in kernels:
        at = "csrc/prt_persist.hip:99:1: remark: "
        lines += [f"{at}Function Name: {name} {B.REMARK}", "   99 |     Params P1) {", "      | ^"]
        lines += [f"{at}    {k}: {v} {B.REMARK}" for k, v in
                  (("TotalSGPRs", 106), ("VGPRs", vgprs), ("ScratchSize [bytes/lane]", 4 * vspill),
                   ("Dynamic Stack", "False"), ("SGPRs Spill", sspill), ("VGPRs Spill", vspill))]
    return "\n".join(lines) + "\n"


PATH2 = ("_Z6k_pathILi1ELb1ELi12ELi341ELi2EEv7Persist6Params", 215, 205, 0)
PATH4 = ("_Z6k_pathILi0ELb1ELi12ELi21ELi4EEv7Persist6Params", 128, 79, 151)
SHADOW = ("_Z8k_shadow6Params", 96, 0, 1)


def test_report_is_read():
    got = B.resource_report("a warning\n" + report([PATH2, SHADOW]))
    assert list(got) == [PATH2[0], SHADOW[0]]
    assert got[PATH2[0]] == {"TotalSGPRs": 106, "VGPRs": 215, "ScratchSize": 0, "SGPRs Spill": 205, "VGPRs Spill": 0}
    assert got[SHADOW[0]]["VGPRs Spill"] == 1


@pytest.mark.parametrize("kernels,ok", [([PATH2, SHADOW], True), ([PATH2, PATH4], False), ([SHADOW], False), ([], False)])
def test_path_kernels_keep_their_registers(kernels, ok):
    if ok:
        B.check_spills(B.resource_report(report(kernels)))
    else:
        with pytest.raises(RuntimeError):
            B.check_spills(B.resource_report(report(kernels)))
