"""The rules that choose a convolution's kernel, tile and grid (csrc/conv_plan.h), compiled for
the host: the plans stay inside what the kernels and a launch can hold, and the cases of the GPU
tests run the code they name."""
import ctypes
import math
import os
import random
import subprocess

import pytest

from ogle_amd import hip as H
import test_kernels_gpu as K

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("plan") / "probe.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "ogle_amd", "csrc"),
                    os.path.join(ROOT, "tests", "conv_plan_probe.cc"), "-o", so], check=True)
    return ctypes.CDLL(so)


def conv(n, h, w, c, o, k=1, s=1, p=0, d=1, g=1, dtype=H.F32):
    """Plan arguments of a convolution; the pointers are only looked at for their alignment."""
    return H.conv_args(4096, 4096, None, 4096, n, h, w, c, o, k, s, p, d, g, H.ACT_NONE, 0.0, 0.0,
                       H.VARIANT_ANY4 if g > 1 else H.VARIANT_NHWC4, dtype)


PATCH_FIELDS = ("cols", "gp", "cc", "runs", "boxes", "box_blocks", "blocks", "vec_x", "vec_w", "lds_floats")


def patch_plan(probe, *shape, **kw):
    out = (ctypes.c_int64 * len(PATCH_FIELDS))()
    if not probe.probe_patch(ctypes.byref(conv(*shape, **kw)), out):
        return None
    return dict(zip(PATCH_FIELDS, out))


def test_infinite_filter_cases_walk_several_boxes(probe):
    """Of the cases with infinite filter values some give a workgroup one box, some several, one
    stages its channels in chunks."""
    args = [(n, h, w, c, o, k, s, p, 1, g) for n, h, w, c, o, k, s, p, g in K.INFINITE_FILTER_CASES]
    assert [probe.probe_direct(ctypes.byref(conv(*a))) for a in args] == [PATCH, PATCH, PATCH, RUNS, PATCH]
    plans = [patch_plan(probe, *a) for a in args[:3] + args[4:]]
    assert [p["boxes"] > p["box_blocks"] for p in plans] == [False, False, True, True]
    assert plans[1]["cc"] < 130
    assert plans[2]["gp"] > 1
    assert plans[3]["runs"] == 1 and plans[3]["cols"] == 64


def random_direct(r):
    """A convolution as the direct kernels may meet it, of any form; None if it has no output."""
    g = r.choice([1, 1, 2, 3, 5, 8, 12, 32])
    k, d, s = r.choice([1, 1, 3, 3, 5, 7, 11]), r.choice([1, 1, 1, 2, 3]), r.choice([1, 1, 2, 3, 4])
    log = lambda lo, hi: int(round(math.exp(r.uniform(math.log(lo), math.log(hi)))))    # noqa: E731
    h, w, p = log(1, 300), log(1, 300), r.choice([0, k // 2, k // 2, k])
    if h + 2 * p < (k - 1) * d + 1 or w + 2 * p < (k - 1) * d + 1:
        return None
    return (log(1, 100), h, w, g * log(1, 200), g * log(1, 200), k, s, p, d, g)


def test_patch_plan_stays_within_lds(probe):
    """A workgroup's dynamic LDS and the kernel's own 16 bytes are at most the 64 KB that a launch
    may ask for; the two pinned shapes fill them but for a few words."""
    for n, h, w, c, o, k, st, p, d, g in K.FULL_LDS_CASES:
        plan = patch_plan(probe, n, h, w, c, o, k, st, p, d, g)
        assert plan is not None and 4 * plan["lds_floats"] + 16 <= 65536
    r, taken, largest = random.Random(5), 0, 0
    for _ in range(20000):
        shape = random_direct(r)
        plan = shape and patch_plan(probe, *shape, dtype=r.choice([H.F32, H.F16]))
        if plan:
            taken += 1
            largest = max(largest, plan["lds_floats"])
            assert 4 * plan["lds_floats"] + 16 <= 65536, shape
    assert taken > 5000 and largest > 16000


def test_patch_plan_stays_within_a_launch(probe):
    """Fewer than 2^32 threads.  The pinned shape, a 1x1 convolution of a padded map whose channels are
    staged in chunks, has one box per workgroup and more of them than that."""
    assert patch_plan(probe, 1, 1000, 1000, 511, 1, 1, 1, 22669) is None
    plan = patch_plan(probe, 1, 1000, 1000, 511, 1, 1, 1, 2000)
    assert plan["cc"] < 511 and plan["boxes"] == plan["blocks"] and plan["blocks"] * 256 < 2 ** 32


GENERAL, PATCH, SMALL_K = 0, 1, 2   # DirectKernel
RUNS = -2                           # none of them: contracted as runs of values


@pytest.mark.parametrize("shape,dtype,kernel", [
    # n, h, w, c, o, k, s, p, d, g: next to the line on both sides, as measured (conv_plan.h); in fp32 most ungrouped,
    # undilated ones are runs by now
    ((1, 1, 1, 17, 33, 3, 1, 1), H.F32, GENERAL),         # eight of nine taps lie in the padding
    ((1, 4, 4, 192, 192, 3, 1, 1, 1, 12), H.F32, PATCH),
    ((1, 14, 14, 7, 33, 3, 1, 1), H.F32, RUNS),
    ((1, 14, 14, 7, 33, 3, 1, 1), H.F16, GENERAL),
    ((1, 14, 14, 17, 33, 3, 1, 1), H.F32, RUNS),
    ((1, 14, 14, 17, 33, 3, 1, 1), H.F16, PATCH),
    ((1, 14, 14, 17, 33, 3, 1, 2, 2), H.F32, PATCH),
    ((1, 56, 56, 35, 33, 1), H.F32, GENERAL),
    ((1, 56, 56, 35, 75, 1), H.F32, RUNS),
    ((1, 56, 56, 35, 75, 1), H.F16, PATCH),
    ((1, 28, 28, 131, 33, 1), H.F32, RUNS),
    ((1, 28, 28, 131, 33, 1), H.F16, GENERAL),
    ((4, 56, 56, 32, 48, 1, 1, 0, 1, 4), H.F32, PATCH),
    ((4, 57, 43, 96, 144, 3, 1, 1, 1, 12), H.F32, PATCH),
])
def test_patch_kernel_where_it_is_faster(probe, shape, dtype, kernel):
    assert probe.probe_direct(ctypes.byref(conv(*shape, dtype=dtype))) == kernel
    assert (patch_plan(probe, *shape, dtype=dtype) is not None) == (kernel == PATCH)


@pytest.mark.parametrize("shape,dtype,kernel", [
    ((1, 1, 1, 33, 16, 3, 1, 1), H.F32, SMALL_K),       # eight of nine taps lie in the padding
    ((1, 14, 14, 7, 16, 3, 1, 1), H.F32, SMALL_K),
    ((1, 14, 14, 17, 16, 3, 1, 1), H.F32, PATCH),
    ((1, 28, 28, 33, 16, 3, 2, 1), H.F16, SMALL_K),     # stride 2: three chunks of channels to stage
    ((1, 56, 56, 35, 64, 1), H.F32, RUNS),
    ((1, 56, 56, 35, 64, 1), H.F16, SMALL_K),
    ((1, 56, 56, 36, 64, 1), H.F16, SMALL_K),
    ((4, 56, 56, 35, 256, 1), H.F32, RUNS),
    ((4, 56, 56, 35, 256, 1), H.F16, PATCH),            # many products
    ((8, 112, 112, 131, 16, 1), H.F32, RUNS),
    ((8, 112, 112, 131, 16, 1), H.F16, PATCH),          # an input of 26 MB
    ((8, 112, 112, 3, 64, 7, 2, 3), H.F32, RUNS),
    ((8, 112, 112, 3, 64, 7, 2, 3), H.F16, PATCH),
    ((1, 14, 14, 28, 256, 1), H.F32, GENERAL),          # short sums of a small output
    ((1, 28, 28, 131, 64, 1), H.F32, RUNS),
    ((1, 28, 28, 131, 64, 1), H.F16, SMALL_K),
    ((1, 28, 28, 12, 16, 3, 1, 1), H.F16, PATCH),
])
def test_direct_kernel_with_the_filter_in_lds(probe, shape, dtype, kernel):
    assert probe.probe_direct(ctypes.byref(conv(*shape, dtype=dtype))) == kernel


@pytest.mark.parametrize("dtype", [H.F32, H.F16])
def test_small_k_cases_run_that_kernel(probe, dtype):
    kernels = [probe.probe_direct(ctypes.byref(conv(*case, dtype=dtype))) for case in K.SMALL_K_CASES]
    assert kernels == [SMALL_K] * 3 + [RUNS if dtype == H.F32 else SMALL_K] * 2 + [SMALL_K]
    threads = [a[0] * a[1] * a[2] * (a[4] // 16) for a in K.SMALL_K_CASES]
    assert min(threads[-2:]) >= 256 * 256 * 4 > max(threads[:-2])


IGEMM_FIELDS = ("bm", "bn", "tiles", "splits", "workspace", "pieces", "rows", "cols")


def igemm_plan(probe, *shape, scratch=True, **kw):
    out = (ctypes.c_int64 * len(IGEMM_FIELDS))()
    if not probe.probe_igemm(ctypes.byref(conv(*shape, **kw)), int(scratch), out):
        return None
    return dict(zip(IGEMM_FIELDS, out))


@pytest.mark.parametrize("shape,pieces", [
    # n, h, w, c, o, k, s, p   fp32 as bf16 pieces: next to the lines (conv_plan.h)
    ((16, 150, 150, 32, 64, 1), False),             # two slabs, 5625 tiles
    ((16, 150, 150, 36, 64, 1), True),              # three
    ((1, 150, 150, 32, 64, 1), False),
    ((1, 128, 128, 128, 128, 1), False),            # 512 workgroups of 8 slabs
    ((1, 128, 128, 144, 128, 1), True),             # of 9
    ((1, 19, 19, 512, 63, 3, 1, 1), False),         # class head of one image: 288 workgroups of 6 slabs
    ((8, 19, 19, 512, 63, 3, 1, 1), True),
    ((1, 189, 189, 512, 24, 1), False),             # pointwise to 24 channels
    ((1, 189, 189, 64, 24, 3, 1, 1), True),
    ((16, 19, 19, 512, 512, 1), True),
])
def test_pieces_where_they_are_faster(probe, shape, pieces):
    assert igemm_plan(probe, *shape)["pieces"] == pieces


def test_large_fp32_tiles_are_pieces(probe):
    """128x128 tiles of fp32 are not built: workgroups of pieces run their plans."""
    r, large = random.Random(7), 0
    for _ in range(40000):
        k = r.choice([1, 1, 3])
        h = int(math.exp(r.uniform(1, 6.5)))
        shape = (r.choice([1, 2, 16, 64]), h, h, 4 * r.choice([2, 3, 4, 8, 9, 12, 16, 64, 128, 256]),
                 r.choice([65, 100, 128, 168, 256, 512, 1024]), k, r.choice([1, 2]), k // 2)
        plan = igemm_plan(probe, *shape, scratch=r.random() < 0.5)
        if plan and (plan["bm"], plan["bn"]) == (128, 128):
            large += 1
            assert plan["pieces"], shape
    assert large > 300


def test_heads_of_one_image_have_no_pieces(probe):
    """So that their grouped launch is the kernel without the code, registers and LDS of pieces."""
    for m, c, a in ((19, 512, 3), (10, 1024, 6), (5, 512, 6), (3, 256, 6), (2, 256, 6), (1, 128, 6)):
        for o in (4 * a, 21 * a):
            assert not igemm_plan(probe, 1, m, m, c, o, 3, 1, 1)["pieces"], (m, o)


@pytest.mark.parametrize("dtype", [H.F32, H.F16])
def test_patch_cases_run_what_they_name(probe, dtype):
    direct = [probe.probe_direct(ctypes.byref(conv(*case, dtype=dtype))) for case in K.PATCH_CASES]
    runs = dtype == H.F32
    assert direct == [PATCH, PATCH, PATCH, -1] + ([RUNS] * 4 if runs else [PATCH, PATCH, GENERAL, PATCH]) + \
        [GENERAL, GENERAL, PATCH, PATCH]
    for case, want in K.PATCH_WIDE_CASES + K.PATCH_NOT_RUNS_CASES:
        plan = patch_plan(probe, *case, dtype=dtype)
        if runs and case == (33, 34, 26, 66, 65, 1, 1, 0, 1, 1):
            assert plan is None and probe.probe_direct(ctypes.byref(conv(*case))) == RUNS
            continue
        assert plan is not None, case
        plan["several"] = plan["boxes"] > plan["box_blocks"]
        assert {key: plan[key] for key in want} == want, (case, plan)
        n, h, w, c, _, k, s, p, d, g = case   # not a stem kernel's
        assert g > 1 or k * k * c > 32 or n * H.out_size(h, k, s, p, d) * H.out_size(w, k, s, p, d) < 4096


def test_pieces_cases_run_what_they_name(probe):
    def tile(*shape, scratch=True):
        plan = igemm_plan(probe, *shape, scratch=scratch)
        name = "%dx%d pieces" % (plan["rows"], plan["cols"]) if plan["pieces"] else "%dx%d" % (plan["bm"], plan["bn"])
        return name + (" split" if plan["splits"] > 1 else "")
    assert [tile(*case) for case in K.PIECES_CASES] == [
        "64x64", "64x64", "64x64 pieces", "128x128 pieces", "128x64 pieces", "32x32", "128x32 pieces", "64x32 pieces",
        "64x64 split", "128x64 pieces", "64x32 pieces", "128x64 pieces", "64x64 pieces split", "64x64"]
    assert [tile(*case, scratch=False) for case in K.PIECES_CASES if tile(*case).endswith("split")] == ["64x32 pieces"] * 2
    assert [tile(3, 75, 75, 512, 64, 3, 1, 1, scratch=False), tile(16, 19, 19, 512, 512, 1),
            tile(1, 160, 160, 32, 256, 3, 1, 1)] == ["128x64 pieces", "64x64 pieces", "128x64 pieces"]
    assert [tile(n, h, w, c, o, k, 1, p) for n, h, w, c, o, k, p in K.NOT_FINITE_CASES] == [
        "64x64 pieces", "128x128 pieces", "64x64 pieces", "128x64 pieces", "64x64 pieces split", "128x32 pieces",
        "128x64 pieces", "64x64"]
    assert [tile(n, h, w, c, o, k, 1, p) for n, h, w, c, o, k, p in K.TINY_CASES] == [
        "64x64 pieces", "128x128 pieces", "128x32 pieces"]
    assert [[tile(*case) for case in batch] for batch in K.BATCHES_OF_PIECES] == [   # each alone
        ["128x64 pieces"] * 2, ["128x32 pieces"] * 2, ["128x64 pieces"] * 2, ["128x64 pieces", "64x64"],
        ["64x64 pieces split", "128x16 split", "64x64", "128x32 pieces"]]


def test_batches_of_one_form(probe):
    """Every form that a grouped launch of one kind has a kernel for is the form of some batch's members."""
    grouped = {4: 1, 5: 1, 6: 8, 7: 8, 2: 10, 9: 11}     # what stands in for a form in a group
    kinds = set()
    for batch in K.BATCHES_OF_PIECES + K.BATCHES_OF_FORMS:
        forms = [probe.probe_form(ctypes.byref(conv(*case)), 1) for case in batch]
        of = {(grouped.get(f, f), case[5] == 1 and case[6] == 1) for f, case in zip(forms, batch)}
        if len(of) == 1 and len(batch) > 1:
            kinds |= of
    assert kinds == {(1, True), (1, False), (3, True), (8, True), (8, False), (10, False), (11, True), (11, False)}


def test_form_cases_run_what_they_name(probe):
    """Every form of the pieces kernel is some case's (PiecesForm, conv_plan.h)."""
    forms = [probe.probe_form(ctypes.byref(conv(*case)), 1) for case, _ in K.FORM_CASES]
    assert forms == [form for _, form in K.FORM_CASES]
    assert set(forms) == set(range(1, 10)) - {8}   # 8 is the K2 forms' in a grouped launch


def test_rows_are_dealt_whole_where_no_unit_gets_another_round(probe):
    """Two workgroups a unit and 32 units an XCD: the fullest XCD has as many rounds as equal shares would give."""
    assert [probe.probe_rows_even(*a) for a in ((100, 5), (83, 6), (169, 3), (65, 4), (96, 5), (64, 4), (163, 3), (1000, 1))] == \
        [0, 0, 0, 0, 1, 1, 1, 1]
    for tiles_m in range(1, 300):
        for per_row in (1, 2, 3, 5, 8):
            if probe.probe_rows_even(tiles_m, per_row):
                most = -(-tiles_m // 8) * per_row
                assert 10 * 8 * -(-tiles_m // 8) <= 11 * tiles_m
                assert most > 512 or -(-most // 64) == -(-(-(-tiles_m * per_row // 8)) // 64)


def test_two_k_groups_where_the_wave_split_kernel_needs_a_second_round(probe):
    """255 and 256 tiles of 32x32: one round; 257 and more: 64x32 tiles in two K groups."""
    forms = [probe.probe_form(ctypes.byref(conv(*shape, 1)), 1)
             for shape in ((2, 28, 29, 256, 154), (1, 32, 32, 256, 256), (1, 33, 32, 256, 256), (3, 31, 31, 312, 96))]
    assert forms == [0, 0, 7, 7]


def test_forms_are_chosen_within_their_tiles(probe):
    """128x128 workgroups and 128x64 ones of four waves are built for pointwise convolutions only, 128x32 ones for others; other types than fp32
    have no form."""
    r, seen = random.Random(11), set()
    for _ in range(30000):
        k = r.choice([1, 1, 3])
        h = int(math.exp(r.uniform(1, 6)))
        shape = (r.choice([1, 2, 16, 64]), h, h, 4 * r.choice([2, 3, 8, 9, 12, 16, 64, 128, 256]),
                 r.choice([12, 31, 40, 65, 100, 128, 168, 256, 512, 1024]), k, r.choice([1, 2]), k // 2)
        form = probe.probe_form(ctypes.byref(conv(*shape)), r.random() < 0.5)
        seen.add(form)
        if form in (3, 4):
            assert k == 1 and shape[6] == 1, shape
        if form == 2:
            assert k == 3 or shape[6] == 2, shape
        if shape[3] % 8 == 0:
            assert probe.probe_form(ctypes.byref(conv(*shape, dtype=H.F16)), 1) <= 0
    assert seen - {-1} == set(range(0, 10)) - {8}


def test_runs_cases_run_what_they_name(probe):
    forms = [probe.probe_runs(ctypes.byref(conv(*case))) for case, _ in K.RUNS_CASES]
    assert forms == [form for _, form in K.RUNS_CASES]
    assert set(forms) == {1, 2, 5, 6, 7, 9}


@pytest.mark.parametrize("shape,kw", [
    ((16, 19, 19, 99, 99, 3, 1, 2, 2), {}),              # dilated
    ((4, 48, 48, 99, 99, 3, 1, 1, 1, 3), {}),            # grouped
    ((4, 56, 56, 99, 99, 3, 1, 1), dict(dtype=H.F16)),
    ((8, 7, 7, 39, 37, 1), {}),                          # short sums of a small output
    ((22, 49, 47, 149, 5, 3, 1, 1), {}),                 # five channels out
    ((1, 1000, 1000, 511, 40, 1, 1, 2000), {}),          # an output beyond 2^31 bytes is fine, padding that long is not
    ((3, 16000, 16000, 3, 64, 7, 2, 3), {}),             # an input beyond 2^31 bytes
])
def test_runs_leave_to_the_direct_kernels(probe, shape, kw):
    assert probe.probe_runs(ctypes.byref(conv(*shape, **kw))) == -1


def test_runs_lose_no_value_at_the_tensors_ends(probe):
    """A vector that begins before the tensor or ends behind it is read value by value if it holds a value of
    the image, in whatever row: all small maps, also those a padding is wider than."""
    shapes = [case for case, _ in K.RUNS_CASES] + [
        (n, h, w, c, 64, k, s, p) for n in (1, 3) for h in (1, 2, 5, 17) for w in (1, 2, 3, 5) for c in (1, 2, 3, 5)
        for k in (1, 2, 3, 5, 7, 15) for s in (1, 2, 3) for p in (0, 1, 3, 7)
        if h + 2 * p >= k and w + 2 * p >= k]
    assert len(shapes) > 3000
    lost = [shape for shape in shapes if probe.probe_runs_lost(ctypes.byref(conv(*shape)))]
    assert not lost, (len(lost), lost[:5])
