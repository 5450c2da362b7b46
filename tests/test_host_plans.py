"""Host-side plans of the H·v kernels (no device): which kernel serves which
call, and how the terms are filed.  host_plans.hip prints the answers."""

import os
import subprocess

import pytest

from hphi_amd import build as B

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    from hphi_amd import capi
    if not os.path.exists(capi.LIB_PATH):
        B.build()
    exe = str(tmp_path_factory.mktemp("plans") / "host_plans")
    lib = os.path.dirname(capi.LIB_PATH)
    subprocess.run([B.HIPCC] + B.HIP_FLAGS + ["--offload-host-only", "-O1", os.path.join(HERE, "host_plans.hip"), "-o", exe,
                                              "-L" + lib, "-lhphi_amd", "-Wl,-rpath," + lib], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return dict(ln.split(" ", 1) for ln in out.splitlines())


@pytest.mark.parametrize("k", [1, 2, 4, 8, 16, 0, -1, 3, 32, 64, 65, 128, 1024, 1028])
def test_class_kernel_serves_its_block_sizes_only(plans, k):
    assert int(plans[f"cls_wanted_{k}"]) == (k in (1, 2, 4, 8, 16))


def test_high_group_is_the_one_the_high_half_pass_applies(plans):
    """The class kernel skips its own high group when the second pass runs; that pass applies the engine's."""
    assert int(plans["hi_wanted"]) == 1 and int(plans["high_terms"]) > 0
    assert int(plans["high_filed_differently"]) == 0


@pytest.mark.parametrize("name,same", [("real_hops", 1), ("complex_hops", 0), ("nn_high", 0), ("assisted", 0)])
def test_lobpcg_runs_by_classes_only_in_the_gather_order(plans, name, same):
    assert int(plans[f"same_order_{name}"]) == same


@pytest.mark.parametrize("k", [1, 8])
def test_autotuner_offers_the_class_kernel_on_a_fresh_engine(plans, k):
    assert int(plans[f"autotune_fresh_{k}"]) == 1


@pytest.mark.parametrize("run,k,on", [("tuned_1_canon", 1, 0), ("tuned_1_lds", 1, 0), ("tuned_1_class4", 1, 1),
                                      ("tuned_1_generic", 1, 0), ("tuned_8_block", 8, 0), ("tuned_8_generic", 8, 0),
                                      ("gc_1_generic", 1, 0), ("gc_2_block", 2, 0), ("gc_8_generic", 8, 0)])
def test_autotuning_one_block_size_leaves_the_others(plans, run, k, on):
    """Whichever kernel wins for k columns, the other block sizes keep theirs and their shape."""
    before, after = plans[run.split("_")[0] + "_none"].split(), plans[run].split()
    assert len(before) == len(after) == 5
    for i in range(5):
        if 1 << i == k:
            assert after[i].startswith(f"{on},")
        else:
            assert after[i] == before[i] and before[i].startswith("1,")


def test_autotuning_leaves_the_best_gather_shape_under_the_class_kernel(plans):
    assert plans["tuned_1_class4"].split()[0] == "1,4"
    assert int(plans["tuned_1_class4_tpb"]) == 512


def test_shapes_set_by_hand_stay_so(plans):
    """k = 1 is the class kernel's; a workgroup size of the block kernel set by hand keeps that kernel for blocks."""
    got = [x.split(",")[0] for x in plans["tuned_1_by_hand"].split()]
    assert got == ["1", "0", "0", "0", "0"]


def test_tiles_without_room_for_their_terms_leave_the_gather_kernels(plans):
    """Neither an error nor tiles."""
    assert plans["tiles_without_memory"].split() == ["0", "0"]


# k = 1, 2, 4, 8, 16: by classes or not; forced for k = 1; at most this many low-half flips
DEFAULTS = {
    "spin_20_2": "1 1 1 1 1", "spin_24_12": "1 1 1 1 1", "spin_24_6": "1 1 1 1 1", "spin_32_6": "1 1 1 1 1",
    "spin_28_5": "1 1 1 1 1",                                  # as dilute, but fewer than 2^17 states
    "spin_30_5": "0 1 1 1 1", "spin_32_27": "0 1 1 1 1",       # dilute: single columns
    "hubbard_4_1_1_0": "0 0 0 1 1", "hubbard_8_1_1_0": "0 0 0 1 1", "hubbard_6_2_2_0": "0 0 1 1 1",  # a few workgroups
    "hubbard_8_3_3_0": "0 1 1 1 1", "hubbard_8_4_4_0": "1 1 1 1 1",
    "hubbard_12_6_6_0": "1 1 1 1 1", "hubbard_16_2_5_0": "1 1 1 1 1",
    "hubbard_14_3_3_0": "0 0 1 1 1", "hubbard_16_3_3_0": "0 0 1 1 1",
    "hubbard_15_3_3_0": "0 0 0 1 1",
    "hubbard_12_6_6_30": "1 1 1 1 1", "hubbard_16_4_4_20": "1 1 1 1 1", "hubbard_16_4_4_32": "1 1 1 1 1",
    "hubbard_12_3_3_30": "0 0 0 0 0",                          # three workgroups per CU, dilute
    "hubbard_16_4_4_36": "0 0 0 0 0",                          # two workgroups per CU
}


@pytest.mark.parametrize("name", DEFAULTS)
def test_default_kernel_of_canonical_sectors(plans, name):
    *wanted, slab, forced, nlo = plans["default_" + name].split()
    assert " ".join(wanted) == DEFAULTS[name], nlo
    assert forced == "1"


# k = 1, 2, 4, 8, 16: in tiles or not
GC_DEFAULTS = {
    "j1j2_18": "0 0 1 1 1", "j1j2_22": "1 1 1 1 1", "hubbard_10": "1 1 1 1 1",
    "pairs_18": "0 0 0 1 1",    # 256 tiles for k = 4, half of the terms of no case
    "pairs_20": "0 0 0 1 1",    # three quarters
    "pairs_22": "1 0 0 1 1",    # the same, 1,024 tiles for k = 1
    "ring_24": "1 1 1 0 0", "hubbard_11": "1 1 1 0 0",  # few terms, blocks of 512 MB
}


@pytest.mark.parametrize("name", GC_DEFAULTS)
def test_default_kernel_of_grand_canonical_sectors(plans, name):
    got = plans["gc_" + name].split()
    assert " ".join(got[:5]) == GC_DEFAULTS[name]
    assert all(f >= w for w, f in zip(got[:5], got[5:])) and "1" in got[5:]


@pytest.mark.parametrize("name,on", [("spin_24_6", 0), ("spin_20_10", 1), ("spin_22_8", 1), ("all_20_10", 0), ("spin_24_12", 1),
                                     ("hubbard_12_5_6_0", 0), ("hubbard_12_6_6_0", 1), ("hubbard_12_6_6_4", 0),
                                     ("hubbard_14_3_3_0", 0), ("all_24_8", 1), ("all_26_7", 0)])
def test_served_slabs_by_classes(plans, name, on):
    """By size, by the share of the states that a term acts on (Hubbard) and by LDS."""
    assert int(plans["default_" + name].split()[5]) == on


@pytest.mark.parametrize("name,ok", [("16_3_200", 1), ("16_3_6000", 0), ("16_8_6000", 1)])
def test_class_layout_keeps_its_target_table_to_a_vector(plans, name, ok):
    """6,000 density-assisted hops on 8,650 blocks: 200 MB of targets for a vector of 5 MB, so none;
    with 8 + 8 electrons the vector is 2.6 GB."""
    assert int(plans["many_terms_" + name]) == ok
