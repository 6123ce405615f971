"""Register and LDS budgets of the kernels whose forms rest on what the compiler holds in registers (staged
loads, values made opaque, loads kept from moving): none spills, and each keeps the wavefronts a SIMD that its
form was chosen for.  Read from the compiler's own metadata as in test_kernel_resources.py."""
import pytest

from test_kernel_resources import HIPCC, LDS_GRANULE, LDS_PER_CU, VGPRS_PER_SIMD_LANE, kernel_metadata, os

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")

# per kernel: wavefronts a SIMD, workgroups a CU whose static LDS has to fit
BUDGETS = {
    "grid_tiled.hip": {"grid_tiled_kernel_small": (6, 2), "9ExactMathELi16ELi16E": (7, 7), "9ExactMathELi15ELi15E": (7, 7),
                       "9ExactMathELi7ELi31E": (7, 7), "8FastMathE": (6, 6)},
    "kernels.hip": {"patch_kernel": (7, 5)},
    "rigid_kernels.hip": {"rigid_step_kernel": (3, 3)},
    "surrogate_kernels.hip": {"sur_mlp_kernelILi2E": (4, 1), "sur_mlp_kernelILi4E": (2, 1), "sur_diag_kernel": (6, 6)},
    "surrogate_train.hip": {"train_chain_kernelILi4E": (1, 1), "train_chain_kernelILi8E": (2, 1),
                            "train_weights_kernel": (2, 2)},
}


@pytest.mark.parametrize("source", sorted(BUDGETS))
def test_no_spills_and_the_occupancy_of_each_form(source, tmp_path):
    kernels = kernel_metadata(source, tmp_path)
    for name, m in kernels.items():
        assert m["vgpr_spill_count"] == 0 and m["private_segment_fixed_size"] == 0, name
    for part, (waves, groups) in BUDGETS[source].items():
        found = {n: m for n, m in kernels.items() if part in n}
        assert found, part
        for name, m in found.items():
            assert VGPRS_PER_SIMD_LANE // (-(-m["vgpr_count"] // 8) * 8) >= waves, (name, m["vgpr_count"])
            lds = -(-m["group_segment_fixed_size"] // LDS_GRANULE) * LDS_GRANULE
            assert groups * lds <= LDS_PER_CU, (name, m["group_segment_fixed_size"])


def test_only_the_exact_forms_that_are_launched_are_built(tmp_path):
    names = kernel_metadata("grid_tiled.hip", tmp_path)
    assert not [n for n in names if "ExactMathELi8ELi8E" in n]
