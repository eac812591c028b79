"""Host-side tests of the launch planner through the C ABI in plan-only mode (include/fastkron_ext.h): every
argument check, the planner and each kernel's check of the concrete buffers run, nothing is launched, no GPU is
needed.  Covered here: which kernels a problem gets, what the launches are handed (strides, batch counts), and the
fallback to plainer kernels when a buffer does not have the alignment a kernel's vector accesses need
(the reference's counterpart is the optimisation level of a kernel, reference src/kernels/kernel_opt.h:42-84,
checked per problem in KMMKernel::canCompute, src/kernels/kmmkernel.cpp:85-126)."""
import ctypes

import pytest

from fastkron_amd import capi

BASE = 0x7000_0000_0000          # fake device addresses, 4 GiB apart; never dereferenced in plan-only mode
GAP = 1 << 32


@pytest.fixture
def planner():
    lib = capi.load()
    h = ctypes.c_void_p()
    assert lib.fastKronInit(ctypes.byref(h), capi.BACKEND_HIP) == capi.SUCCESS
    assert lib.fastKronSetPlanOnly(h, 1) == capi.SUCCESS
    yield lib, h
    lib.fastKronDestroy(h)


@pytest.fixture
def online_planner(monkeypatch):
    """A plan-only handle without the shipped tuned plans: the online rules alone."""
    monkeypatch.setenv("FASTKRON_SHIPPED_PLANS", "0")
    lib = capi.load()
    h = ctypes.c_void_p()
    assert lib.fastKronInit(ctypes.byref(h), capi.BACKEND_HIP) == capi.SUCCESS
    assert lib.fastKronSetPlanOnly(h, 1) == capi.SUCCESS
    yield lib, h
    lib.fastKronDestroy(h)


def plan(planner, mm, dt, M, Ps, Qs, batch=None, alpha=1.0, beta=0.0, with_y=False, offs=None, strides=None,
         strideF=None, opX=capi.OP_N, opF=capi.OP_N, temp2=True, y_is_z=False):
    """Runs one call in plan-only mode.  `offs` shifts the fake base pointers of x / z / y / t1 / t2 by bytes,
    `strides` overrides the element strides of x / z / y.  Returns (error, kernel names, launch records)."""
    lib, h = planner
    offs = offs or {}
    K, L = 1, 1
    for p, q in zip(Ps, Qs):
        K, L = K * p, L * q
    ptr = {n: BASE + i * GAP + offs.get(n, 0) for i, n in enumerate(["x", "z", "y", "t1", "t2"])}
    if y_is_z:
        ptr["y"] = ptr["z"]
    fs = capi.arr_ptr([BASE + (8 + i) * GAP + offs.get("f", 0) for i in range(len(Ps))])
    sc = ctypes.c_float if dt == "s" else ctypes.c_double
    X, Z = ctypes.c_void_p(ptr["x"]), ctypes.c_void_p(ptr["z"])
    Y = ctypes.c_void_p(ptr["y"]) if (with_y or y_is_z) else None
    t1, t2 = ctypes.c_void_p(ptr["t1"]), (ctypes.c_void_p(ptr["t2"]) if temp2 else None)
    PsA, QsA = capi.arr_u32(Ps), capi.arr_u32(Qs)
    if batch is None:
        if mm == "mkm":
            e = getattr(lib, dt + "gemkm")(h, capi.BACKEND_HIP, M, len(Ps), PsA, QsA, X, opX, fs, opF, Z, sc(alpha), sc(beta),
                                           Y, t1, t2)
        else:
            e = getattr(lib, dt + "gekmm")(h, capi.BACKEND_HIP, len(Ps), QsA, PsA, M, fs, opF, X, opX, Z, sc(alpha), sc(beta),
                                           Y, t1, t2)
    else:
        st = {"x": M * K, "z": M * L, "y": M * L}
        st.update(strides or {})
        sF = capi.arr_u64(strideF if strideF is not None else [p * q for p, q in zip(Ps, Qs)])
        if mm == "mkm":
            e = getattr(lib, dt + "gemkmStridedBatched")(h, capi.BACKEND_HIP, M, len(Ps), PsA, QsA, X, opX, st["x"], fs, opF,
                                                         sF, Z, st["z"], sc(alpha), sc(beta), batch, Y, st["y"], t1, t2)
        else:
            e = getattr(lib, dt + "gekmmStridedBatched")(h, capi.BACKEND_HIP, len(Ps), QsA, PsA, M, fs, opF, sF, X, opX,
                                                         st["x"], Z, st["z"], sc(alpha), sc(beta), batch, Y, st["y"], t1, t2)
    buf = ctypes.create_string_buffer(1 << 16)
    lib.fastKronGetLastPlan(h, buf, len(buf))
    names = [s.split(":")[1] for s in buf.value.decode().split(";")[1:]]
    lib.fastKronGetLastLaunches(h, buf, len(buf))
    launches = []
    for line in buf.value.decode().splitlines():
        rec = dict(kv.split("=", 1) for kv in line.split())
        rec["f_batch"] = [int(v) for v in rec["f_batch"].split(",")]
        launches.append(rec)
    return e, names, launches


# ---- a strided-batched call with one batch entry must not carry its strides into any launch ----
@pytest.mark.parametrize("dt,M,P,N", [("s", 8, 16, 5), ("s", 4, 8, 6), ("s", 2, 32, 4), ("d", 8, 16, 4), ("d", 2, 64, 3),
                                      ("s", 16, 4, 8), ("d", 4, 8, 5), ("s", 4, 12, 4)])
def test_single_entry_batches_carry_no_strides(planner, dt, M, P, N):
    e, names, launches = plan(planner, "mkm", dt, M, [P] * N, [P] * N, batch=1)
    assert e == capi.SUCCESS
    assert len(launches) >= 1
    for rec in launches:
        assert rec["f_batch"] == [0] * len(rec["f_batch"]), (names, rec)
    # ... and it gets the plan of the plain entry point
    e2, names2, launches2 = plan(planner, "mkm", dt, M, [P] * N, [P] * N)
    assert e2 == capi.SUCCESS and names2 == names
    assert [r["batch"] for r in launches2] == [r["batch"] for r in launches]


def test_two_part_plan_reads_leading_factors_with_stride_zero(planner):
    """M rows become batch entries of the leading part: per-entry factor strides there would walk off F."""
    e, names, launches = plan(planner, "mkm", "s", 8, [16] * 5, [16] * 5, batch=1)
    assert e == capi.SUCCESS and len(launches) == 2
    assert "_16x16_16x16_4_1x65536" in launches[0]["kernel"] and int(launches[0]["M"]) == 8 * 16
    assert int(launches[1]["batch"]) == 8 and launches[1]["f_batch"] == [0]
    # per-batch leading factors rule the two-part plan out altogether
    e, names, launches = plan(planner, "mkm", "s", 8, [16] * 5, [16] * 5, batch=2)
    assert e == capi.SUCCESS
    assert all(int(r["batch"]) == 2 for r in launches), launches
    # shared factors (stride 0) with several batch entries keep it
    e, names, launches = plan(planner, "mkm", "s", 8, [16] * 5, [16] * 5, batch=2, strideF=[0] * 5)
    assert e == capi.SUCCESS and int(launches[-1]["batch"]) == 16 and launches[-1]["f_batch"] == [0]


def test_fp64_rows_of_five_8x8_factors_get_the_whole_row_kernel(online_planner):
    """dgemkm 8x8^5 from 32 rows on: one launch of the fp64 row kernel on the chain as given (no 64x64 products); with
    fewer rows, with eight factors or in the KMM layout the chain is merged as before."""
    row = "mkm_hip_gfx950_512_d_8x8_8x8_5_1x32768_valu_NN_strided_0_3"
    for M, opF in [(1024, capi.OP_N), (32, capi.OP_T)]:
        e, names, launches = plan(online_planner, "mkm", "d", M, [8] * 5, [8] * 5, opF=opF, beta=0.5, with_y=True)
        assert e == capi.SUCCESS and names == [row], names
    e, names, _ = plan(online_planner, "mkm", "d", 31, [8] * 5, [8] * 5)
    assert e == capi.SUCCESS and row not in names and any("64x64" in n for n in names), names
    # six or seven factors: the row kernel on the blocks of 32768 columns, the leading factor(s) across the blocks
    e, names, launches = plan(online_planner, "mkm", "d", 1024, [8] * 6, [8] * 6)
    assert e == capi.SUCCESS and len(names) == 2 and names[0] == row and int(launches[0]["M"]) == 8192, (names, launches)
    e, names, launches = plan(online_planner, "mkm", "d", 16, [8] * 7, [8] * 7)
    assert e == capi.SUCCESS and len(names) == 2 and names[0] == row and "64x64" in names[1], names
    e, names, _ = plan(online_planner, "mkm", "d", 3, [8] * 6, [8] * 6)           # 24 blocks: merged as before
    assert e == capi.SUCCESS and row not in names and any("64x64" in n for n in names), names
    e, names, _ = plan(online_planner, "mkm", "d", 16, [8] * 8, [8] * 8)
    assert e == capi.SUCCESS and row not in names, names
    e, names, _ = plan(online_planner, "kmm", "d", 1024, [8] * 5, [8] * 5)
    assert e == capi.SUCCESS and row not in names, names
    # per-batch factors: every batch entry reads its own five factors
    e, names, launches = plan(online_planner, "mkm", "d", 16, [8] * 5, [8] * 5, batch=4)
    assert e == capi.SUCCESS and names == [row] and launches[0]["f_batch"] == [64] * 5, (names, launches)


def test_rows_of_three_32x32_factors_choose_the_kernel_by_row_count(online_planner):
    """sgemkm 32x32^3: from three rows per CU on the persistent kernel (one workgroup of 16 waves per CU), from 96 rows on
    the kernel with two workgroups of 8 waves per CU, below that the pair kernel and a step; the same on the blocks of
    a longer chain."""
    pers = "mkm_hip_gfx950_1024_f_32x32_32x32_3_1x32768_mfma16x16x4_NN_strided_0_3"
    two = "mkm_hip_gfx950_512_f_32x32_32x32_3_1x32768_mfma16x16x4_NN_strided_0_3"
    for M, want in [(1024, [pers]), (768, [pers]), (767, [two]), (96, [two])]:
        e, names, _ = plan(online_planner, "mkm", "s", M, [32] * 3, [32] * 3, beta=0.5, with_y=True)
        assert e == capi.SUCCESS and names == want, (M, names)
    e, names, _ = plan(online_planner, "mkm", "s", 95, [32] * 3, [32] * 3)
    assert e == capi.SUCCESS and pers not in names and two not in names and len(names) == 2, names
    e, names, launches = plan(online_planner, "mkm", "s", 24, [32] * 4, [32] * 4)          # 768 blocks
    assert e == capi.SUCCESS and names[0] == pers and int(launches[0]["M"]) == 768, (names, launches)
    e, names, _ = plan(online_planner, "mkm", "s", 96, [32] * 3, [32] * 3, batch=8)         # 768 rows in all
    assert e == capi.SUCCESS and names == [pers], names
    # a misaligned operand sends both away (16-byte accesses)
    e, names, _ = plan(online_planner, "mkm", "s", 1024, [32] * 3, [32] * 3, offs={"x": 4})
    assert e == capi.SUCCESS and pers not in names and two not in names, names


def test_rectangular_pairs_get_the_pair_kernel_and_the_two_part_plan(online_planner):
    """Two 32x64 / 64x32 factors: one launch on exact tiles; three: the pair on the blocks of a row (M * P virtual rows of
    P*P columns, Q*Q out) and the leading factor across the blocks as a KMM problem with one batch entry per row."""
    for dt, P, Q in [("s", 32, 64), ("s", 64, 32), ("d", 32, 64)]:
        name = f"mkm_hip_gfx950_256_{'f' if dt == 's' else 'd'}_{P}x{Q}_{P}x{Q}_2_1x{P * P}_mfma16x16x4_NN_strided_0_3"
        e, names, launches = plan(online_planner, "mkm", dt, 40, [P] * 2, [Q] * 2, beta=0.5, with_y=True)
        assert e == capi.SUCCESS and names == [name], names
        e, names, launches = plan(online_planner, "mkm", dt, 3, [P] * 3, [Q] * 3, beta=0.5, with_y=True)
        assert e == capi.SUCCESS and len(names) == 2 and names[0] == name, names
        assert int(launches[0]["M"]) == 3 * P and int(launches[0]["out"], 16) == BASE + 3 * GAP, launches      # into temp1
        assert int(launches[1]["M"]) == Q * Q and int(launches[1]["batch"]) == 3, launches
        assert int(launches[1]["in"], 16) == BASE + 3 * GAP and int(launches[1]["out"], 16) == BASE + 1 * GAP, launches
    # fp64 64x32 has no such kernel (a 64 x 64 tile of doubles per row in flight): one launch per factor
    e, names, _ = plan(online_planner, "mkm", "d", 40, [64] * 2, [32] * 2)
    assert e == capi.SUCCESS and len(names) == 2 and all("_2_1x" not in n for n in names), names
    # the leading factors of a two-part plan are shared between the rows: per-batch factors rule it out
    e, names, _ = plan(online_planner, "mkm", "s", 3, [32] * 3, [64] * 3, batch=2)
    assert e == capi.SUCCESS and len(names) == 3, names


def test_pairs_of_64x64_fp64_factors_by_block_count(online_planner):
    """dgemkm 64x64^2: the pair kernel from 8 blocks per CU on (a block per wave) and between 1.25 and 4 blocks per CU
    (a block shared by waves); otherwise two single steps."""
    pair = "mkm_hip_gfx950_512_d_64x64_64x64_2_1x4096_mfma4x4x4_NN_strided_0_3"
    for M, fused in [(256, False), (319, False), (320, True), (512, True), (1024, True), (1025, False), (2047, False),
                     (2048, True), (16384, True)]:
        e, names, _ = plan(online_planner, "mkm", "d", M, [64] * 2, [64] * 2)
        assert e == capi.SUCCESS and (names == [pair]) == fused and len(names) == (1 if fused else 2), (M, names)
    e, names, launches = plan(online_planner, "mkm", "d", 8, [64] * 3, [64] * 3)            # 512 blocks of a longer chain
    assert e == capi.SUCCESS and names[0] == pair and int(launches[0]["M"]) == 512, (names, launches)


# ---- kernels with 16-byte global accesses are only chosen for buffers that allow them ----
VECTOR_CASES = [
    # (label, mm, dt, M, Ps, Qs, batch, beta, substring of the kernel expected on aligned buffers)
    ("row16x4", "mkm", "s", 128, [16] * 4, [16] * 4, None, 0.5, "_16x16_16x16_4_1x65536"),
    ("row16x3", "mkm", "s", 64, [16] * 3, [16] * 3, None, 0.5, "_16x16_16x16_3_1x4096"),
    ("row16x3d", "mkm", "d", 64, [16] * 3, [16] * 3, None, 0.5, "_d_16x16_16x16_3_1x4096"),
    ("row32x3", "mkm", "s", 128, [32] * 3, [32] * 3, None, 0.5, "_32x32_32x32_3_1x32768"),
    ("pair32", "mkm", "s", 64, [32] * 2, [32] * 2, None, 0.5, "_32x32_32x32_2_1x1024"),
    ("pair64d", "mkm", "d", 2048, [64] * 2, [64] * 2, None, 0.5, "_d_64x64_64x64_2_1x4096"),
    ("step64", "mkm", "s", 64, [64], [64], None, 0.5, "_64x64_64x64_1_"),
    ("kmm64d", "kmm", "d", 64, [64], [64], 8, 0.5, "kmm_hip_gfx950_256_d_64x64_64x64_1_64x64"),
    ("row8x5", "mkm", "s", 64, [8] * 5, [8] * 5, None, 0.5, "_8x8_8x8_5_1x32768"),
    ("row32x16", "mkm", "s", 64, [32] * 3, [16] * 3, None, 0.5, "_32x16_32x16_3_1x32768"),
    ("kmm4x6", "kmm", "s", 1032, [4] * 6, [4] * 6, None, 0.5, "_4x4_4x4_6_8x4096"),
    ("kmm4x6 two-phase", "kmm", "s", 2048, [4] * 6, [4] * 6, None, 0.5, "_4x4_4x4_6_256x4096"),
    ("wide128", "mkm", "s", 8, [128] * 2, [128] * 2, None, 0.5, "_128x128_128x128_1_1x4096_mfma16x16x4lds"),
    ("wide64k", "kmm", "s", 64, [64] * 2, [64] * 2, None, 0.5, "_64x64_64x64_1_64x64_mfma16x16x4lds"),
]


@pytest.mark.parametrize("case", VECTOR_CASES, ids=[c[0] for c in VECTOR_CASES])
def test_aligned_buffers_get_the_specialised_kernel(planner, case):
    _, mm, dt, M, Ps, Qs, batch, beta, want = case
    e, names, _ = plan(planner, mm, dt, M, Ps, Qs, batch=batch, beta=beta, with_y=True)
    assert e == capi.SUCCESS
    assert any(want in n for n in names), names


@pytest.mark.parametrize("which", ["x", "z", "y"])
@pytest.mark.parametrize("case", VECTOR_CASES, ids=[c[0] for c in VECTOR_CASES])
def test_a_buffer_off_by_one_element_still_gets_a_plan_that_accepts_it(planner, case, which):
    """The base pointer of X, Z or Y is moved by one element: whatever plan comes back passed every kernel's own
    check of these buffers (plan-only mode runs them), and the call does not fail."""
    _, mm, dt, M, Ps, Qs, batch, beta, want = case
    esize = 4 if dt == "s" else 8
    e, names, launches = plan(planner, mm, dt, M, Ps, Qs, batch=batch, beta=beta, with_y=True, offs={which: esize})
    assert e == capi.SUCCESS and len(launches) >= 1, names


VECTOR_KERNELS_NEEDING = {
    # kernels whose 16-byte accesses make them refuse a misaligned operand: label -> operands they vector-access
    "row16x4": "xzy", "row16x3": "x", "row16x3d": "x", "row32x3": "xzy", "pair32": "x", "pair64d": "xzy", "step64": "x",
    "kmm64d": "xzy", "wide128": "xzy", "wide64k": "xzy",
}


@pytest.mark.parametrize("label,which", [(k, w) for k, ws in VECTOR_KERNELS_NEEDING.items() for w in ws])
def test_misaligned_operand_rules_the_vector_kernel_out(planner, label, which):
    case = [c for c in VECTOR_CASES if c[0] == label][0]
    _, mm, dt, M, Ps, Qs, batch, beta, want = case
    esize = 4 if dt == "s" else 8
    e, names, _ = plan(planner, mm, dt, M, Ps, Qs, batch=batch, beta=beta, with_y=True, offs={which: esize})
    assert e == capi.SUCCESS
    assert not any(want in n for n in names), (which, names)


@pytest.mark.parametrize("label", ["row16x4", "row32x3", "pair64d", "row16x3"])
@pytest.mark.parametrize("which", ["x", "z", "y"])
def test_odd_batch_strides_rule_the_vector_kernel_out(planner, label, which):
    """Batch entries one element further apart than the operand is long: entry 1 is misaligned although entry 0 is not."""
    case = [c for c in VECTOR_CASES if c[0] == label][0]
    _, mm, dt, M, Ps, Qs, _, beta, want = case
    K, L = 1, 1
    for p, q in zip(Ps, Qs):
        K, L = K * p, L * q
    odd = {"x": M * K + 1, "z": M * L + 1, "y": M * L + 1}[which]
    e, names, launches = plan(planner, mm, dt, M, Ps, Qs, batch=3, beta=beta, with_y=True, strides={which: odd},
                              strideF=[0] * len(Ps))
    assert e == capi.SUCCESS
    needs = VECTOR_KERNELS_NEEDING[label]
    if which in needs:
        assert not any(want in n for n in names), (which, names)


def test_batches_beyond_one_grid_dimension_are_checked_chunk_by_chunk(planner):
    e, names, launches = plan(planner, "mkm", "s", 1, [16, 16], [16, 16], batch=70000, strideF=[0, 0])
    assert e == capi.SUCCESS
    assert [int(r["batch"]) for r in launches] == [65535, 70000 - 65535] * (len(launches) // 2)
    first, second = launches[0], launches[1]
    assert int(second["in"], 16) - int(first["in"], 16) == 65535 * 256 * 4


# ---- tuned-plan files are not trusted ----
def test_tuned_plans_that_do_not_fit_the_problem_are_ignored(planner, tmp_path):
    lib, h = planner
    e, online, _ = plan(planner, "mkm", "s", 8, [8, 8, 8], [8, 8, 8])
    generic = "gekmm_hip_gfx950_256_f_generic_1"
    key = "8x512*(8x8^3)_NN_f"
    bad = [
        f"{key} 0.01 1 0 5 {generic}",                       # factor index beyond the chain
        f"{key} 0.01 2 2 2 {generic} 0 0 {generic}",         # factor 1 never applied
        f"{key} 0.01 3 0 0 {generic} 1 1 {generic} 2 2 {generic}",   # first factor first
        f"{key} 0.01 1 0 2 {generic}",                       # a one-factor kernel given three factors
        f"{key} 0.01 1 0 2 mkm_hip_gfx950_1024_f_16x16_16x16_4_1x65536_mfma16x16x4_NN_strided_0_3",   # wrong factor size
    ]
    for line in bad:
        f = tmp_path / "tuned.db"
        f.write_text(line + "\n")
        assert lib.fastKronSetTunedDB(h, str(f).encode()) == capi.SUCCESS
        e, names, _ = plan(planner, "mkm", "s", 8, [8, 8, 8], [8, 8, 8])
        assert e == capi.SUCCESS and names == online, line
    good = f"{key} 0.01 3 2 2 {generic} 1 1 {generic} 0 0 {generic}"
    f = tmp_path / "tuned.db"
    f.write_text(good + "\n")
    lib.fastKronSetTunedDB(h, str(f).encode())
    e, names, _ = plan(planner, "mkm", "s", 8, [8, 8, 8], [8, 8, 8])
    assert e == capi.SUCCESS and names == [generic] * 3


# ---- op(X) = T: a transposed copy of X ahead of the launches when that saves passes over the data ----
def test_transposed_x_is_copied_first_when_the_whole_row_kernels_then_apply(planner):
    e, names, launches = plan(planner, "mkm", "s", 64, [8] * 5, [8] * 5, opX=capi.OP_T)
    assert e == capi.SUCCESS
    assert names[0].startswith("transpose_") and "_8x8_8x8_5_1x32768" in names[1] and len(names) == 2, names
    # the launches read the copy (temp2), not X
    assert int(launches[0]["in"], 16) == BASE + 4 * GAP
    # the same for the two-part plan of a longer chain and for GeKMM
    e, names, _ = plan(planner, "mkm", "s", 8, [16] * 5, [16] * 5, opX=capi.OP_T)
    assert e == capi.SUCCESS and names[0].startswith("transpose_") and len(names) == 3, names
    # GeKMM with 64x64 factors (with small factors it runs as a GeMKM, below)
    e, names, _ = plan(planner, "kmm", "s", 64, [64] * 2, [64] * 2, opX=capi.OP_T)
    assert e == capi.SUCCESS and names[0].startswith("transpose_") and names[0].endswith("_x") and len(names) == 3, names


def test_gekmm_with_transposed_x_runs_as_the_gemkm_of_that_buffer(online_planner):
    """op(X) = T in a GeKMM means the buffer holds M x K, the X of a GeMKM with transposed factors: the whole-row GeMKM
    kernels run on it, their result goes to temp1 and one transposition (with beta * Y) writes Z."""
    planner = online_planner
    e, names, launches = plan(planner, "kmm", "s", 64, [8] * 5, [8] * 5, opX=capi.OP_T, beta=0.5, with_y=True)
    assert e == capi.SUCCESS and "mkm_" in names[0] and "_8x8_8x8_5_1x32768" in names[0] and names[-1].endswith("_z"), names
    assert len(names) == 2 and len(launches) == 1
    # the launch reads the caller's X, writes temp1, and leaves alpha in and beta * Y out
    assert int(launches[0]["in"], 16) == BASE and int(launches[0]["out"], 16) == BASE + 3 * GAP
    assert launches[0]["y"] == "(nil)"
    # a longer chain: the two-part GeMKM plan, with temp2 and Z as its temporaries
    e, names, launches = plan(planner, "kmm", "s", 1024, [8] * 6, [8] * 6, opX=capi.OP_T)
    assert e == capi.SUCCESS and len(names) == 3 and names[-1].endswith("_z"), names
    assert int(launches[-1]["out"], 16) == BASE + 3 * GAP
    # Y in place (Y == Z, beta != 0): Z cannot serve as a temporary
    e, names, launches = plan(planner, "kmm", "s", 1024, [8] * 6, [8] * 6, opX=capi.OP_T, beta=1.0, y_is_z=True)
    assert e == capi.SUCCESS and names[-1].endswith("_z"), names
    assert all(int(r["out"], 16) != BASE + GAP for r in launches), launches
    # 64x64 factors and larger only with fewer than 64 columns (and fp64 chains of three 64x64 factors)
    e, names, _ = plan(planner, "kmm", "s", 1024, [64] * 2, [64] * 2, opX=capi.OP_T)
    assert e == capi.SUCCESS and not names[-1].endswith("_z"), names
    e, names, _ = plan(planner, "kmm", "s", 16, [128] * 3, [128] * 3, opX=capi.OP_T)
    assert e == capi.SUCCESS and names[-1].endswith("_z"), names
    e, names, _ = plan(planner, "kmm", "d", 256, [64] * 3, [64] * 3, opX=capi.OP_T)
    assert e == capi.SUCCESS and names[-1].endswith("_z"), names
    e, names, _ = plan(planner, "kmm", "d", 16, [8] * 5, [8] * 5, opX=capi.OP_T)
    assert e == capi.SUCCESS and names[-1].endswith("_z"), names
    # X not transposed: only large fp32 problems with fewer than 64 columns go this way, X transposed into temp2 first
    e, names, launches = plan(planner, "kmm", "s", 16, [8] * 8, [8] * 8)
    assert e == capi.SUCCESS and names[0].endswith("_x") and names[-1].endswith("_z") and len(names) == 4, names
    assert int(launches[0]["in"], 16) == BASE + 4 * GAP and int(launches[-1]["out"], 16) == BASE + 3 * GAP, launches
    e, names, _ = plan(planner, "kmm", "s", 48, [16] * 4, [16] * 4)
    assert e == capi.SUCCESS and not names[-1].endswith("_z"), names
    e, names, _ = plan(planner, "kmm", "d", 16, [8] * 8, [8] * 8)
    assert e == capi.SUCCESS and not names[-1].endswith("_z"), names
    # rectangular factors stay on the GeKMM kernels
    e, names, _ = plan(planner, "kmm", "s", 256, [32] * 3, [16] * 3, opX=capi.OP_T)
    assert e == capi.SUCCESS and not names[-1].endswith("_z"), names


@pytest.mark.parametrize("dt,M,Ps,opX", [("d", 3, [5] * 7, capi.OP_T), ("d", 73, [6, 4, 2, 8, 7], capi.OP_T), ("s", 16, [16] * 5, capi.OP_N)])
@pytest.mark.parametrize("own", [False, True])
def test_gekmm_as_a_gemkm_leaves_what_lies_between_the_entries_of_z(online_planner, dt, M, Ps, opX, own):
    """Z is a temporary of the GeMKM only where its entries lie side by side; otherwise other results may lie between them."""
    L = 1
    for p in Ps:
        L *= p
    es = 4 if dt == "s" else 8
    for gap in (0, 8, 4 * M * L):
        e, names, launches = plan(online_planner, "kmm", dt, M, Ps, Ps, batch=5, opX=opX, strideF=None if own else [0] * len(Ps),
                                  strides={"z": M * L + gap})
        assert e == capi.SUCCESS
        z = BASE + GAP                                                          # (x, z, y, t1, t2)
        written = [int(l["out"], 16) for l in launches]
        inZ = [w for w in written if z <= w < z + 5 * (M * L + gap) * es]
        assert gap == 0 or not names[-1].startswith("transpose_") or not inZ, (names, launches)


def test_transposed_x_is_read_in_place_when_a_copy_does_not_pay_or_does_not_fit(planner):
    # one small factor: the plain kernel reads the transposed X directly, a copy would add a pass
    e, names, _ = plan(planner, "mkm", "s", 64, [8], [8], opX=capi.OP_T)
    assert e == capi.SUCCESS and not any(n.startswith("transpose_") for n in names), names
    # shrinking chain: X (M x 32768) is larger than a temporary (M x 16384)
    e, names, _ = plan(planner, "mkm", "s", 64, [32] * 3, [16] * 3, opX=capi.OP_T)
    assert e == capi.SUCCESS and not any(n.startswith("transpose_") for n in names), names
    # no second temporary and a plan of several launches: temp1 cannot hold the copy
    e, names, _ = plan(planner, "mkm", "s", 8, [16] * 5, [16] * 5, opX=capi.OP_T, temp2=False)
    assert e == capi.SUCCESS and not any(n.startswith("transpose_") for n in names), names
    # no second temporary but a single launch: the copy goes to temp1
    e, names, launches = plan(planner, "mkm", "s", 64, [8] * 5, [8] * 5, opX=capi.OP_T, temp2=False)
    assert e == capi.SUCCESS and names[0].startswith("transpose_") and len(names) == 2, names
    assert int(launches[0]["in"], 16) == BASE + 3 * GAP


def test_copy_into_the_only_temporary_is_decided_on_every_calls_own_buffers(online_planner):
    """Without a second temporary the transposed copy of X sits in temp1, so the launches behind it must be one launch.
    How many they are depends on the buffers of the call at hand: a second call of the same shape whose temp1 (or Z) is
    off the alignment of the whole-row kernel gets several launches and must then read the transposed X in place;
    no launch may ever read and write the same buffer."""
    for dt, M, P, N in [("s", 1024, 16, 4), ("s", 1024, 64, 2), ("d", 1024, 32, 2)]:
        e, names, launches = plan(online_planner, "mkm", dt, M, [P] * N, [P] * N, opX=capi.OP_T, temp2=False)
        assert e == capi.SUCCESS and names[0].startswith("transpose_") and len(names) == 2, (dt, P, names)
        for offs in ({"t1": 4}, {"z": 4}, {"t1": 4, "z": 4}):
            e, names, launches = plan(online_planner, "mkm", dt, M, [P] * N, [P] * N, opX=capi.OP_T, temp2=False, offs=offs)
            assert e == capi.SUCCESS, (dt, P, offs)
            for rec in launches:
                assert rec["in"] != rec["out"], (dt, P, offs, names, rec)
            if any(n.startswith("transpose_") for n in names):
                assert len(names) == 2, (dt, P, offs, names)
        # and the aligned call still gets the copy afterwards
        e, names, _ = plan(online_planner, "mkm", dt, M, [P] * N, [P] * N, opX=capi.OP_T, temp2=False)
        assert e == capi.SUCCESS and names[0].startswith("transpose_") and len(names) == 2, (dt, P, names)


def test_leaving_plan_only_mode_drops_its_stand_in_workspace():
    """Plan-only mode on a handle without a device uses a stand-in address for the merged-factor workspace; once the
    mode is left, a call must not plan on it (it would be handed to kernels): without a device and a workspace the
    chain is then not merged, and fastKronInitHIP allocates the real one."""
    lib = capi.load()
    h = ctypes.c_void_p()
    assert lib.fastKronInit(ctypes.byref(h), capi.BACKEND_HIP) == capi.SUCCESS
    try:
        assert lib.fastKronSetPlanOnly(h, 1) == capi.SUCCESS
        e, names, _ = plan((lib, h), "mkm", "s", 1024, [4] * 8, [4] * 8)
        assert e == capi.SUCCESS and len(names) == 1 and "16x16" in names[0], names       # merged into 16x16^4
        assert lib.fastKronSetPlanOnly(h, 0) == capi.SUCCESS
        assert lib.fastKronSetPlanOnly(h, 1) == capi.SUCCESS
        e, names, _ = plan((lib, h), "mkm", "s", 1024, [4] * 8, [4] * 8)
        assert e == capi.SUCCESS and len(names) == 1 and "16x16" in names[0], names       # the stand-in is back, as before
    finally:
        lib.fastKronDestroy(h)


def test_transposition_rules_that_came_from_tuned_plans(online_planner):
    planner = online_planner
    copied = lambda names: names[0].startswith("transpose_")
    # a padded-step first launch on a 128-wide factor counts twice in the MKM layout, also with 16 rows ...
    e, names, _ = plan(planner, "mkm", "s", 16, [128] * 3, [128] * 3, opX=capi.OP_T)
    assert e == capi.SUCCESS and copied(names) and len(names) == 4, names
    # ... in the KMM layout only while X is at most 64 MB
    e, names, _ = plan(planner, "kmm", "s", 1024, [128] * 2, [128] * 2, opX=capi.OP_T)
    assert e == capi.SUCCESS and copied(names), names
    e, names, _ = plan(planner, "kmm", "s", 320, [128] * 3, [128] * 3, opX=capi.OP_T)
    assert e == capi.SUCCESS and not copied(names) and len(names) == 3, names
    # equal launch counts: the copy goes first, except in the KMM layout with fewer than 64 columns
    e, names, _ = plan(planner, "mkm", "d", 256, [16] * 4, [16] * 4, opX=capi.OP_T)
    assert e == capi.SUCCESS and copied(names), names
    e, names, _ = plan(planner, "kmm", "d", 16, [16] * 6, [16] * 6, opX=capi.OP_T)
    assert e == capi.SUCCESS and not copied(names), names


# ---- online rules for chains outside the specialised kernels ----
def test_lds_fused_groups_get_balanced_depth(online_planner):
    """The LDS-fused kernel taken as deep as it goes would leave a single plain launch (or two): the last two groups share
    the factors about equally instead."""
    planner = online_planner
    e, names, _ = plan(planner, "mkm", "s", 1024, [2] * 7, [4] * 7)
    assert e == capi.SUCCESS and len(names) == 2 and all("small_fused" in n for n in names), names
    e, names, _ = plan(planner, "kmm", "s", 1024, [3] * 7, [3] * 7)
    assert e == capi.SUCCESS and len(names) == 2 and all("small_fused" in n for n in names), names
    # a chain that one group holds stays one launch
    e, names, _ = plan(planner, "mkm", "s", 1024, [3] * 7, [3] * 7)
    assert e == capi.SUCCESS and len(names) == 1 and "small_fused" in names[0], names


def test_whole_rows_of_small_square_factors_run_in_place(online_planner):
    """One launch where the factors cover whole rows of at most 160 KB, are square and X is not transposed; few long rows in
    passes of one digit stay with the kernel that spreads a row over workgroups."""
    def inplace(mm, dt, M, Ps, Qs=None, **kw):
        e, names, _ = plan(online_planner, mm, dt, M, Ps, Qs or Ps, **kw)
        assert e == capi.SUCCESS
        return len(names) == 1 and "inplace" in names[0]
    mixed = [2, 3, 4, 5, 6, 7, 8]
    for dt in ("s", "d"):
        assert inplace("mkm", dt, 1, [5] * 6) and inplace("mkm", dt, 1001, [5] * 6, beta=0.5, with_y=True)
        assert inplace("mkm", dt, 7, [7, 3, 8], opF=capi.OP_T, offs={"x": 4 if dt == "s" else 8, "z": 8})
        assert inplace("mkm", dt, 9, [5, 5, 5], batch=3) and inplace("kmm", dt, 1, [5] * 4)
        assert not inplace("mkm", dt, 9, [5, 5, 5], opX=capi.OP_T) and not inplace("kmm", dt, 2, [5] * 4)
        assert not inplace("mkm", dt, 9, [5, 5], [5, 4]) and not inplace("mkm", dt, 9, [5] * 7)
    assert not inplace("mkm", "s", 95, mixed) and inplace("mkm", "s", 96, mixed)
    assert not inplace("mkm", "d", 95, [7] * 5) and inplace("mkm", "d", 96, [7] * 5) and inplace("mkm", "s", 1, [7] * 5)
    assert not inplace("mkm", "d", 1000, mixed)                       # 315 KB

    # longer rows: blocks of as many trailing factors as the kernel holds, at most two factors across the blocks
    def blocks(dt, M, Ps, **kw):
        e, names, launches = plan(online_planner, "mkm", dt, M, Ps, Ps, **kw)
        assert e == capi.SUCCESS
        return int(launches[0]["M"]) if "inplace" in names[0] and int(launches[0]["lo"]) == 0 and len(names) > 1 else None
    assert blocks("s", 3, [5] * 7) == 15 and blocks("d", 3, [5] * 8) == 75 and blocks("s", 2, [6] * 6) == 12
    assert blocks("s", 1, [7] * 6) == 7 and blocks("s", 2, [9, 2] + [3] * 8) == 36 and blocks("s", 9, [5] * 7, beta=0.5, y_is_z=True) == 45
    assert blocks("s", 3, [3] * 11) is None and blocks("s", 3, [64] + [5] * 3) is None      # three leading ones; short blocks
    assert blocks("d", 34, [6] * 6) is None and blocks("d", 35, [6] * 6) == 210      # (the measured crossing)
    assert blocks("d", 13, [7] * 6) is None and blocks("d", 14, [7] * 6) == 98 and blocks("d", 32, [2, 2] + [6] * 5) is None
    assert blocks("s", 3, [5] * 7, batch=2) is None and blocks("s", 3, [5] * 7, batch=2, strideF=[0] * 7) == 15


def test_padded_step_rules_for_rectangular_and_large_odd_factors(online_planner):
    planner = online_planner
    # shrinking factors with 16 rows: padded matrix-core step, not the plain kernel
    for dt in ("s", "d"):
        e, names, _ = plan(planner, "mkm", dt, 1024, [16] * 5, [8] * 5)
        assert e == capi.SUCCESS and len(names) == 5 and all("anyxany" in n for n in names), names
    # fp64, KMM layout, more than 128 rows: plain kernel when the padded groups of four stay part empty
    e, names, _ = plan(planner, "kmm", "d", 1024, [129] * 2, [129] * 2)
    assert e == capi.SUCCESS and all("generic" in n for n in names), names
    e, names, _ = plan(planner, "kmm", "d", 1024, [255] * 2, [255] * 2)
    assert e == capi.SUCCESS and all("anyxany" in n for n in names), names
    e, names, _ = plan(planner, "kmm", "s", 1024, [200] * 2, [200] * 2)
    assert e == capi.SUCCESS and all("anyxany" in n for n in names), names


# ---- the plans that ship with the library (fastkron_amd/gfx950_plans.txt) ----
def _parse_key(key):
    """'MxK*(PxQ^N)_NN_f' / '(PxQ^N)*KxM_TT_d' (factor lists as 'AxB(x)CxD') -> (mm, dt, M, Ps, Qs, opX, opF)."""
    import re
    m = re.match(r"^(\d+)x(\d+)\*\((.*)\)_([NT])([NT])_([fd])$", key)
    if m:
        mm, M, facs, ox, of, dt = "mkm", int(m.group(1)), m.group(3), m.group(4), m.group(5), m.group(6)
    else:
        m = re.match(r"^\((.*)\)\*(\d+)x(\d+)_([NT])([NT])_([fd])$", key)
        assert m, key
        mm, M, facs, ox, of, dt = "kmm", int(m.group(3)), m.group(1), m.group(4), m.group(5), m.group(6)
    Ps, Qs = [], []
    for f in facs.split("(x)"):
        pq, _, n = f.partition("^")
        p, q = pq.split("x")
        Ps += [int(p)] * int(n or 1)
        Qs += [int(q)] * int(n or 1)
    op = {"N": capi.OP_N, "T": capi.OP_T}
    return mm, ("s" if dt == "f" else "d"), M, Ps, Qs, op[ox], op[of]


def _shipped_records():
    import os
    path = os.path.join(os.path.dirname(capi.LIB_PATH), "..", "gfx950_plans.txt")
    recs = []
    for line in open(path):
        if line.startswith("#") or not line.strip():
            continue
        tok = line.split()
        i = 2
        flags = {}
        while tok[i][0] in "MSX":
            flags[tok[i][0]] = int(tok[i][1:])
            i += 1
        n = int(tok[i])
        steps = [(int(tok[i + 1 + 3 * k]), int(tok[i + 2 + 3 * k]), tok[i + 3 + 3 * k]) for k in range(n)]
        recs.append((tok[0], flags, steps))
    return recs


def test_every_shipped_plan_is_what_a_default_handle_runs(planner):
    recs = _shipped_records()
    assert len(recs) >= 3
    for key, flags, steps in recs:
        if "stridedBatched" in key:
            continue
        mm, dt, M, Ps, Qs, opX, opF = _parse_key(key)
        e, names, launches = plan(planner, mm, dt, M, Ps, Qs, opX=opX, opF=opF)
        assert e == capi.SUCCESS, key
        want = [k for _, _, k in steps]
        got = [n for n in names if not n.startswith("transpose_")]
        assert got == want, (key, names, want)
        assert any(n.startswith("transpose_") for n in names) == bool(flags.get("X", 0)), (key, names)


def test_shipped_plans_can_be_switched_off(monkeypatch):
    """FASTKRON_SHIPPED_PLANS=0: a handle created then selects online, as if the file were not there."""
    import ctypes
    recs = [r for r in _shipped_records() if "stridedBatched" not in r[0]]
    monkeypatch.setenv("FASTKRON_SHIPPED_PLANS", "0")
    lib = capi.load()
    h = ctypes.c_void_p()
    assert lib.fastKronInit(ctypes.byref(h), capi.BACKEND_HIP) == capi.SUCCESS
    assert lib.fastKronSetPlanOnly(h, 1) == capi.SUCCESS
    try:
        differ = 0
        for key, flags, steps in recs:
            mm, dt, M, Ps, Qs, opX, opF = _parse_key(key)
            e, names, _ = plan((lib, h), mm, dt, M, Ps, Qs, opX=opX, opF=opF)
            assert e == capi.SUCCESS
            got = [n for n in names if not n.startswith("transpose_")]
            differ += got != [k for _, _, k in steps] or any(n.startswith("transpose_") for n in names) != bool(flags.get("X", 0))
        assert differ == len(recs)          # every record is there because tuning beat the online plan
    finally:
        lib.fastKronDestroy(h)


# ---- non-temporal hints: what a launch is told about its input and output ----
def _hints(launches):
    return [(int(r["stream_in"]), int(r["stream_out"])) for r in launches]


def test_large_cold_operands_are_streamed(planner):
    """One launch over 134 MB in and out (sgemkm 1024 x 8^5): both hints; the same call on 256 rows: none."""
    e, names, launches = plan(planner, "mkm", "s", 1024, [8] * 5, [8] * 5)
    assert e == capi.SUCCESS and len(launches) == 1 and _hints(launches) == [(1, 1)]
    e, names, launches = plan(planner, "mkm", "s", 256, [8] * 5, [8] * 5)
    assert e == capi.SUCCESS and _hints(launches) == [(0, 0)]


def test_intermediates_that_fit_the_memory_side_cache_are_not_streamed(planner):
    """sgemkm 128 x 8^6 runs two launches around an intermediate of 134 MB: the first launch streams X in but stores
    ordinarily, the second loads ordinarily and streams Z out.  With 256 rows (268 MB) everything is streamed."""
    e, names, launches = plan(planner, "mkm", "s", 128, [8] * 6, [8] * 6)
    assert e == capi.SUCCESS and len(launches) == 2 and _hints(launches) == [(1, 0), (0, 1)]
    e, names, launches = plan(planner, "mkm", "s", 256, [8] * 6, [8] * 6)
    assert e == capi.SUCCESS and len(launches) == 2 and _hints(launches) == [(1, 1), (1, 1)]


def test_a_transposed_copy_is_not_streamed_back_in(planner):
    """op(X) = T behind a transposed copy: the copy (134 MB) was written a moment ago, so the launch that reads it
    loads ordinarily."""
    e, names, launches = plan(planner, "mkm", "s", 1024, [8] * 5, [8] * 5, opX=capi.OP_T, opF=capi.OP_T)
    assert e == capi.SUCCESS and names[0].startswith("transpose_") and len(launches) == 1
    assert _hints(launches) == [(0, 1)]


def test_two_part_plans_keep_their_intermediate_ordinary(planner):
    """sgemkm 16 x 16^6 (two-part plan, 1 GB per buffer): beyond the cache everything streams; 2 x 16^5 (8 MB): nothing."""
    e, names, launches = plan(planner, "mkm", "s", 2, [16] * 5, [16] * 5)
    assert e == capi.SUCCESS and all(h == (0, 0) for h in _hints(launches))
    e, names, launches = plan(planner, "mkm", "s", 32, [16] * 5, [16] * 5)     # 134 MB per buffer
    assert e == capi.SUCCESS and len(launches) >= 2
    hints = _hints(launches)
    assert hints[0][0] == 1 and hints[-1][1] == 1                  # X in and Z out are streamed
    assert all(h[1] == 0 for h in hints[:-1]) and all(h[0] == 0 for h in hints[1:])   # nothing in between is


def test_a_small_result_behind_a_large_input_is_streamed_out(planner):
    """8 x 512 x (32x16)^3 with Y: 537 MB of X, 67 MB of Z; the launch moves far more than the caches hold."""
    e, names, launches = plan(planner, "mkm", "s", 512, [32] * 3, [16] * 3, batch=8, beta=1.0, with_y=True)
    assert e == capi.SUCCESS and len(launches) == 1 and _hints(launches) == [(1, 1)]


# ---- a kernel that refuses the call's buffers is replaced by the next one in line ----
@pytest.mark.parametrize("which,expect", [("z", "_128x128_128x128_1_1x2048_mfma16x16x4_NN"), ("y", "_128x128_128x128_1_1x2048_mfma16x16x4_NN"),
                                          ("x", "anyxany")])
def test_a_refusing_kernel_is_replaced_by_the_next_in_line(planner, which, expect):
    """sgemkm 8 x 128^2: the wide step kernel needs X, Z and Y on 16-byte boundaries, the streaming step only X, the
    padded step nothing: an operand one element off moves the plan down that list, not to the plain kernel."""
    e, names, launches = plan(planner, "mkm", "s", 8, [128] * 2, [128] * 2, beta=0.5, with_y=True, offs={which: 4})
    assert e == capi.SUCCESS and len(launches) == 2
    assert all(expect in n for n in names), names


@pytest.mark.parametrize("mm", ["mkm", "kmm"])
@pytest.mark.parametrize("opX", [capi.OP_N, capi.OP_T])
def test_gradient_functions_launch_nothing_in_plan_only_mode(planner, mm, opX):
    """Without a GPU any launch, and any look at the device, would be an error."""
    lib, h = planner
    M, Ps, Qs = 6, [3, 4, 8], [5, 4, 8]
    shape = (int(mm == "mkm"), 0, M, 3, capi.arr_u32(Ps), capi.arr_u32(Qs))
    save, work = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib.fastKronGradSizes(h, *shape, opX, M * 96, 1, 2, ctypes.byref(save), ctypes.byref(work)) == capi.SUCCESS
    ptr = [ctypes.c_void_p(BASE + i * GAP) for i in range(8)]
    fs, gf = (capi.arr_ptr([BASE + (n + i) * GAP for i in range(3)]) for n in (10, 13))
    args = (h, *shape, ptr[0], opX, M * 96, fs, capi.OP_N, 1, 2)
    assert lib.fastKronGradForward(*args, ptr[1], ptr[2]) == capi.SUCCESS
    buf = ctypes.create_string_buffer(1 << 14)
    lib.fastKronGetLastLaunches(h, buf, len(buf))
    assert [l.split()[1] for l in buf.value.decode().splitlines()] == ["lo=2", "lo=1", "lo=0"]
    assert lib.fastKronGradBackward(*args, ptr[3], ptr[2], ptr[4], gf, ptr[5]) == capi.SUCCESS
    lib.fastKronGetLastLaunches(h, buf, len(buf))
    assert [l.split()[0] for l in buf.value.decode().splitlines()] == ["kernel=gradient_step"] * 3 + ["kernel=gradient_sum"]
    assert lib.fastKronGradBackward(*args, None, ptr[2], ptr[4], gf, ptr[5]) != capi.SUCCESS


@pytest.mark.parametrize("P,Q", [(96, 192), (192, 96), (192, 192), (384, 384), (640, 640), (100, 100), (512, 512), (64, 64), (33, 40), (2048, 128)])
@pytest.mark.parametrize("batch", [1, 5])
def test_workgroups_of_the_backward_kernel_come_in_multiples_of_the_cus(planner, P, Q, batch):
    """Workgroups of one launch for a factor's gradient (64x64 blocks of it, by partial sums, by batch entries) on 256 CUs, with
    rows enough for any number of them: at least three quarters of the places they take are filled."""
    lib, h = planner
    M = 2 ** 20
    shape = (0, 0, M, 1, capi.arr_u32([P]), capi.arr_u32([Q]))
    ptr = [ctypes.c_void_p(BASE + i * GAP) for i in range(8)]
    one = lambda i: capi.arr_ptr([BASE + i * GAP])
    assert lib.fastKronGradBackward(h, *shape, ptr[0], capi.OP_N, M * P, one(10), capi.OP_N, 1, batch, ptr[3], ptr[2], None, one(11),
                                    ptr[5]) == capi.SUCCESS
    buf = ctypes.create_string_buffer(1 << 14)
    lib.fastKronGetLastLaunches(h, buf, len(buf))
    step = dict(kv.split("=") for kv in buf.value.decode().splitlines()[0].split())
    groups = int(step["sums"]) * -(-P // 64) * -(-Q // 64) * batch
    places = -(-groups // 256) * 256
    assert groups >= 0.75 * places, (groups, places)


def test_gekmm_chains_of_small_factors_keep_their_digits_in_place(online_planner):
    """Groups of equal small factors as problems on the columns behind them: their row counts, strides and batch entries; other
    plans where factors differ per entry, X has gaps, or as many launches of the register kernels do."""
    def groups(dt, M, Ps, **kw):
        e, names, launches = plan(online_planner, "kmm", dt, M, Ps, Ps, **kw)
        assert e == capi.SUCCESS
        return [(int(l["M"]), int(l["batch"])) for l in launches] if any("columns" in n for n in names) else None
    for dt in ("s", "d"):
        assert groups(dt, 88, [7] * 6) == [(88, 343), (88 * 343, 1)]
        assert groups(dt, 10, [7] * 6, batch=3, strideF=[0] * 6) == [(10, 3 * 343), (10 * 343, 3)]
        assert groups(dt, 10, [7] * 6, batch=3) is None                                          # factors of each entry's own
        assert groups(dt, 10, [7] * 6, batch=3, strideF=[0] * 6, strides={"x": 10 * 7 ** 6 + 8}) is None
        assert groups(dt, 10, [7] * 3, batch=3) == [(10, 3)]                                      # whole problems: own factors as well
        assert groups(dt, 5, [6, 6, 16, 3, 3, 3]) == [(5, 576), (5 * 27, 36), (5 * 432, 1)]
        assert groups(dt, 9, [5] * 7, beta=0.5, y_is_z=True) == [(9, 125), (9 * 625, 1)]
        assert groups(dt, 9, [5] * 9, temp2=False) is None                                       # three groups need two temporaries
    assert groups("s", 1024, [8] * 5) is None and groups("s", 2048, [4] * 6) is None
    assert groups("d", 16, [16] * 3) is None and groups("d", 3, [9, 9]) is None


PAIR = "_anyxany_64x64_2_1xany_"


@pytest.mark.parametrize("dt,M,a,b,pair", [
    # one launch (us against the two steps): few rows always, many where a row is enough work
    ("s", 1, (31, 63), (31, 63), True), ("s", 256, (2, 2), (9, 9), True), ("s", 1100, (50, 40), (12, 20), True), ("d", 2500, (33, 17), (9, 12), True),
    ("d", 1003, (31, 63), (31, 63), True), ("d", 515, (48, 64), (48, 64), True),
    # the two steps: dgemkm 203 / 41, 82 / 45, sgemkm 53 / 33, and the kernel with two LDS buffers 35.7 / 14.8
    ("d", 251160, (2, 2), (9, 9), False), ("d", 7300, (3, 20), (43, 57), False), ("s", 7038, (8, 8), (64, 64), False), ("d", 44884, (2, 10), (7, 5), False)])
def test_two_factors_are_one_launch_where_that_is_faster(online_planner, dt, M, a, b, pair):
    for opF in (capi.OP_N, capi.OP_T):
        e, names, _ = plan(online_planner, "mkm", dt, M, [a[0], b[0]], [a[1], b[1]], opF=opF)
        assert e == capi.SUCCESS and any(PAIR in n for n in names) == pair, names


@pytest.mark.parametrize("dt,M,a,b,copied", [
    # sgemkm 59 / 144 and 15 / 18 with the copy; 33 / 19, 15.5 / 13.9 and 11.3 / 9.6 with it, without
    ("s", 7936, (62, 62), (20, 20), True), ("s", 26247, (14, 14), (12, 12), True), ("d", 6685, (2, 1), (32, 40), False), ("s", 284, (33, 33), (33, 33), False),
    ("s", 40, (33, 33), (50, 50), False), ("s", 100, (31, 31), (31, 31), True)])
def test_transposed_x_is_copied_for_the_pair_only_where_that_is_faster(online_planner, dt, M, a, b, copied):
    e, names, _ = plan(online_planner, "mkm", dt, M, [a[0], b[0]], [a[1], b[1]], opX=capi.OP_T)
    assert e == capi.SUCCESS and names[0].startswith("transpose_") == copied, names


def test_padded_pairs_of_many_rows_name_the_kernel_that_runs(planner, tmp_path):
    """Equal factors of 17x17 ... 31x31 on 2048 rows and more, fp32: the pair of any sizes by rule, the padded pair by record."""
    padded = "mkm_hip_gfx950_256_f_32x32_32x32_2_1x1024_mfma16x16x4_NN_strided_0_3"
    for P in (17, 20, 24, 31):
        for dt, M, batch, any_size in [("s", 2047, None, False), ("s", 2048, None, True), ("s", 30000, None, True), ("s", 700, 3, True), ("d", 30000, None, False)]:
            e, names, _ = plan(planner, "mkm", dt, M, [P] * 2, [P] * 2, batch=batch)
            assert e == capi.SUCCESS and len(names) == 1 and ((PAIR if any_size else "_32x32_32x32_2_1x1024_") in names[0]), (P, dt, M, names)
    lib, h = planner
    db = tmp_path / "plans.txt"
    db.write_text(f"5000x576*(24x24^2)_NN_f 0.01 M0 S0 1 0 1 {padded}\n")
    lib.fastKronSetTunedDB(h, str(db).encode())
    e, names, _ = plan(planner, "mkm", "s", 5000, [24] * 2, [24] * 2)
    assert e == capi.SUCCESS and names == [padded]


# ---- products with two batch dimensions ----
def outer_plan(planner, mm, dt, M, Ps, Qs, count, opX=capi.OP_N, opF=capi.OP_N, sx=None, sz=None, beta=0.0, y_is_z=False):
    """fastKronProductOuter in plan-only mode; the strides are those of compact operands unless sx gives X's."""
    lib, h = planner
    K, L = 1, 1
    for p, q in zip(Ps, Qs):
        K, L = K * p, L * q
    ptr = [ctypes.c_void_p(BASE + i * GAP) for i in range(5)]            # x, z, y, t1, t2
    fs = capi.arr_ptr([BASE + (8 + i) * GAP for i in range(len(Ps))])
    sz = capi.arr_u64(sz if sz is not None else [count[1] * M * L, M * L])
    e = lib.fastKronProductOuter(h, mm == "mkm", dt == "d", M, len(Ps), capi.arr_u32(Ps), capi.arr_u32(Qs), ptr[0], opX,
                                 capi.arr_u64(sx if sx is not None else [count[1] * M * K, M * K]), fs, opF, ptr[1], sz, 1.0, beta,
                                 capi.arr_u32(count), (ptr[1] if y_is_z else ptr[2]) if beta else None, sz, ptr[3], ptr[4])
    buf = ctypes.create_string_buffer(1 << 16)
    lib.fastKronGetLastPlan(h, buf, len(buf))
    names = [s.split(":")[1] for s in buf.value.decode().split(";")[1:]]
    lib.fastKronGetLastLaunches(h, buf, len(buf))
    launches = []
    for line in buf.value.decode().splitlines():
        rec = dict(kv.split("=", 1) for kv in line.split())
        rec["f_batch"] = [int(v) for v in rec["f_batch"].split(",")]
        launches.append(rec)
    return e, names, launches


@pytest.mark.parametrize("mm,dt,M,P,N", [("kmm", "s", 88, 7, 6), ("kmm", "d", 16, 8, 5), ("mkm", "s", 8, 16, 5), ("mkm", "d", 2, 64, 3),
                                         ("mkm", "s", 1, 31, 3), ("kmm", "s", 5, 9, 4)])
def test_one_entry_of_two_dimensions_is_the_plain_call(online_planner, mm, dt, M, P, N):
    """Blocks of one problem's rows become batch entries of a launch: no stride of the caller's may reach them."""
    plain = plan(online_planner, mm, dt, M, [P] * N, [P] * N)
    e, names, launches = outer_plan(online_planner, mm, dt, M, [P] * N, [P] * N, (1, 1))
    assert e == plain[0] == capi.SUCCESS and names == plain[1]
    for rec in launches:
        assert rec["f_batch"] == [0] * len(rec["f_batch"]), rec
    # one entry of factors for several of X: the batch with shared factors
    shared = plan(online_planner, mm, dt, M, [P] * N, [P] * N, batch=3, strideF=[0] * N)
    e, names, launches = outer_plan(online_planner, mm, dt, M, [P] * N, [P] * N, (3, 1))
    assert e == shared[0] == capi.SUCCESS and names == shared[1]
    assert [r["batch"] for r in launches] == [r["batch"] for r in shared[2]]
    assert all(r["f_batch"] == [0] * len(r["f_batch"]) for r in launches)


@pytest.mark.parametrize("count,sx,outer_in,entries", [((2, 3), "shared", 0, 1), ((2, 3), "own", None, 6), ((2, 3), "outer", None, 2)])
def test_transposed_copies_of_two_dimensions_are_those_that_are_read(online_planner, count, sx, outer_in, entries):
    """X of op T in front of the rows of five 8x8 factors is copied first: as many entries as differ, and the launch reads those."""
    M, K = 32, 8 ** 5
    strides = {"shared": [0, 0], "own": [count[1] * M * K, M * K], "outer": [M * K, 0]}[sx]
    e, names, launches = outer_plan(online_planner, "mkm", "s", M, [8] * 5, [8] * 5, count, opX=capi.OP_T, sx=strides)
    assert e == capi.SUCCESS and names[0].startswith("transpose_") and len(launches) == 1, (names, launches)
    rec = launches[0]
    lib, h = online_planner
    buf = ctypes.create_string_buffer(1 << 12)
    lib.fastKronGetLastPlan(h, buf, len(buf))
    copied = buf.value.decode().split(";")[0].split("_stridedBatched_")[1]                # the problem whose X is copied
    assert int(rec["batch"]) == count[0] * count[1] and int(rec["inner"]) == count[1] and int(copied) == entries
    # the last entry that the launch reads is the last one that the copy has written
    last = (count[0] - 1) * int(rec["outer_in"]) + (count[1] - 1) * int(rec["in_batch"])
    assert last == (entries - 1) * M * K and (outer_in is None or int(rec["outer_in"]) == outer_in), rec


@pytest.mark.parametrize("mm,dt,M,P,N,count,opX,series", [
    # launches of the series (all entries) against the loop's: us series / loop 374 / 143, 505 / 257, 649 / 264, 174 / 89, 179 / 101
    ("mkm", "s", 460, 14, 3, (10, 4), capi.OP_N, False), ("kmm", "s", 50, 7, 5, (9, 7), capi.OP_N, False), ("kmm", "d", 2, 7, 6, (39, 3), capi.OP_N, False),
    ("mkm", "d", 245, 11, 3, (8, 5), capi.OP_N, False), ("kmm", "s", 2, 8, 6, (8, 3), capi.OP_N, False), ("mkm", "s", 17, 12, 5, (4, 3), capi.OP_N, False),
    # 41 / 54, 85 / 164, one launch either way, and a copy ahead of both
    ("mkm", "s", 32, 13, 3, (19, 3), capi.OP_N, True), ("mkm", "d", 20, 11, 3, (25, 9), capi.OP_N, True), ("mkm", "s", 1001, 5, 6, (2, 3), capi.OP_N, True),
    ("mkm", "s", 32, 8, 5, (2, 3), capi.OP_T, True), ("mkm", "d", 5, 12, 2, (2, 3), capi.OP_N, True), ("mkm", "s", 3, 5, 3, (2, 3), capi.OP_N, True)])
def test_two_dimensions_are_one_series_where_that_is_no_slower(online_planner, mm, dt, M, P, N, count, opX, series):
    K = M * P ** N
    perF = count[0] > count[1]                        # the loop's calls: one entry of factors with all of X, or one of X with all factors
    for _ in range(2):                                # decided, and remembered
        e, names, launches = outer_plan(online_planner, mm, dt, M, [P] * N, [P] * N, count, opX=opX, sx=[K, 0])
        assert e == capi.SUCCESS and all(("inner" in l) == series for l in launches), names
        if series:
            assert all(int(l["batch"]) == count[0] * count[1] for l in launches)
        else:
            plain = plan(online_planner, mm, dt, M, [P] * N, [P] * N, batch=max(count), strideF=[0] * N if perF else None,
                         strides={"x": K if perF else 0, "z": (count[1] if perF else 1) * K})
            assert names == plain[1] and [l["batch"] for l in launches] == [l["batch"] for l in plain[2]]


@pytest.mark.parametrize("dt,M,P,N", [("s", 64, 10, 4), ("s", 16, 9, 5)])
def test_two_dimensions_with_the_factors_outside_are_the_calls_with_shared_factors(online_planner, dt, M, P, N):
    """X of (12) entries and factors of (3, 1): three calls, whose entries lie without gaps, in two parts each."""
    K = M * P ** N
    shared = plan(online_planner, "mkm", dt, M, [P] * N, [P] * N, batch=12, strideF=[0] * N)
    e, names, launches = outer_plan(online_planner, "mkm", dt, M, [P] * N, [P] * N, (12, 3), sx=[K, 0], sz=[K, 12 * K])
    assert e == capi.SUCCESS and names == shared[1] and all("inner" not in l for l in launches), names


def test_records_of_the_loops_calls_are_what_two_dimensions_run(online_planner, tmp_path):
    lib, h = online_planner
    generic = "gekmm_hip_gfx950_256_f_generic_1"
    e, names, launches = outer_plan(online_planner, "mkm", "s", 32, [13] * 2, [13] * 2, (19, 3), sx=[32 * 169, 0])
    assert e == capi.SUCCESS and "inner" in launches[0]
    f = tmp_path / "plans.txt"
    f.write_text(f"32x169*(13x13^2)_NN_f_stridedBatched_19_Fs3 0.01 M0 S0 2 1 1 {generic} 0 0 {generic}\n")
    lib.fastKronSetTunedDB(h, str(f).encode())
    e, names, launches = outer_plan(online_planner, "mkm", "s", 32, [13] * 2, [13] * 2, (19, 3), sx=[32 * 169, 0])
    assert e == capi.SUCCESS and names == [generic] * 2 and all(l["batch"] == "19" and "inner" not in l for l in launches), launches


def test_two_dimensions_without_entries_are_refused(online_planner):
    """As a strided batch of no entries is."""
    for count in [(3, 0), (0, 3), (1, 0), (0, 0)]:
        e, _, _ = outer_plan(online_planner, "mkm", "s", 4, [8, 8], [8, 8], count)
        assert e == capi.INVALID_KMM_PROBLEM, count


def test_gekmm_of_small_factors_runs_as_a_gemkm_where_that_is_faster(online_planner):
    """fp32, few columns, 64 MB of X and more: no equal neighbours, or batches whose factors or gaps rule the groups out, in six
    launches and more or on 8 to 23 columns (2 x 17 columns of 4x3x7x6x3x6x5x6x4 551 us, 688 without)."""
    def via(M, Ps, **kw):
        e, names, _ = plan(online_planner, "kmm", "s", M, Ps, Ps, **kw)
        assert e == capi.SUCCESS
        return names[0].startswith("transpose_") and names[-1].startswith("transpose_")
    mixed, equal = [4, 3, 7, 6, 3, 6, 5, 6, 4], [7] * 7
    assert via(17, mixed) and via(17, mixed, batch=2) and via(17, mixed, batch=2, strideF=[0] * 9)
    assert not via(30, equal) and not via(30, equal, batch=2, strideF=[0] * 7)
    assert via(30, equal, batch=2) and via(30, equal, batch=2, strideF=[0] * 7, strides={"x": 30 * 7 ** 7 + 32})
    assert not via(4, [7] * 8, batch=4) and not via(63, [3, 4, 4, 6, 4, 6, 4, 2, 7], batch=3)


def test_a_last_factor_of_its_own_keeps_the_digits_in_place_only_with_columns_enough(online_planner):
    """Us with the groups against without: 643 / 222, 153 / 65, 121 / 44; 51 / 75 (few entries), 0.7 to 0.9 (many columns)."""
    def inplace(dt, M, Ps, **kw):
        e, names, launches = plan(online_planner, "kmm", dt, M, Ps, Ps, **kw)
        assert e == capi.SUCCESS
        return int(launches[0]["batch"]) > kw.get("batch", 1)
    assert not inplace("s", 2, [8, 7, 7, 7, 12, 12, 12]) and not inplace("d", 5, [8, 3, 7, 7, 7, 6, 3], batch=2, strideF=[0] * 7)
    assert not inplace("s", 6, [8, 8, 6, 7, 4, 7, 3]) and not inplace("s", 47, [6, 7, 7, 2, 3, 3, 7, 6, 2])
    assert inplace("s", 6, [7, 7, 7, 10]) and inplace("d", 10, [7, 7, 7, 10]) and inplace("s", 300, [7, 7, 7, 7, 7, 3])


@pytest.mark.parametrize("dt,M,P,batch,own,opX,pair", [
    ("d", 8056, 36, 1, False, capi.OP_N, False), ("d", 1900, 36, 1, False, capi.OP_N, True), ("d", 1000, 42, 6, False, capi.OP_N, False),
    ("d", 1000, 42, 6, True, capi.OP_N, True), ("s", 2467, 45, 3, True, capi.OP_N, True),
    ("d", 9710, 39, 1, False, capi.OP_T, True)])                                                # 216 us behind a copy, 338 without
def test_pairs_of_33_to_47_rows_a_side_end_where_the_padded_step_reads_whole_pieces(online_planner, dt, M, P, batch, own, opX, pair):
    e, names, _ = plan(online_planner, "mkm", dt, M, [P] * 2, [P] * 2, batch=batch if batch > 1 else None, strideF=None if own else [0] * 2, opX=opX)
    assert e == capi.SUCCESS and any(PAIR in n for n in names) == pair, names


@pytest.mark.parametrize("M,P,Q,opX,pair", [(242, 6, 50, capi.OP_N, False), (60, 6, 50, capi.OP_N, True), (1071, 7, 28, capi.OP_N, False),
                                            (200, 50, 50, capi.OP_N, True), (7, 7, 44, capi.OP_T, True)])
def test_trailing_pairs_leave_no_long_rows_to_the_plain_step(online_planner, M, P, Q, opX, pair):
    """fp64, from 1024 blocks on: leading factors whose rows grow stay with the padded step, but behind a transposed copy."""
    N = 4 if opX == capi.OP_T else 3
    e, names, _ = plan(online_planner, "mkm", "d", M, [P] * N, [Q] * N, opX=opX)
    assert e == capi.SUCCESS and any(PAIR in n for n in names) == pair, names


@pytest.mark.parametrize("dt,M,a,b,batch,pair", [("d", 1, 32, 64, 8, False), ("d", 235, 64, 32, 1, False), ("d", 235, 16, 64, 1, True),
                                                 ("s", 235, 24, 64, 1, True)])
def test_pairs_of_32_and_64_in_fp64_are_two_exact_steps(online_planner, dt, M, a, b, batch, pair):
    e, names, _ = plan(online_planner, "mkm", dt, M, [a, b], [a, b], batch=batch if batch > 1 else None, strideF=[0] * 2)
    assert e == capi.SUCCESS and any(PAIR in n for n in names) == pair, names


@pytest.mark.parametrize("dt,M,P,copied", [("s", 7304, 9, False), ("s", 2653, 11, False), ("d", 3963, 9, False), ("s", 60000, 12, True), ("d", 60000, 12, True)])
def test_small_transposed_x_of_small_factors_is_read_as_it_is_stored(online_planner, dt, M, P, copied):
    e, names, _ = plan(online_planner, "mkm", dt, M, [P] * 2, [P] * 2, opX=capi.OP_T)
    assert e == capi.SUCCESS and names[0].startswith("transpose_") == copied, names


def test_copies_of_a_transposed_x_are_not_made_for_one_row(online_planner):
    """A row is stored the same either way: where the copy's plan is the better one it runs on X itself."""
    for dt, Ps in [("d", [57] * 4), ("s", [6, 36, 6]), ("s", [8] * 5), ("s", [16] * 4)]:
        plain = plan(online_planner, "mkm", dt, 1, Ps, Ps)
        e, names, launches = plan(online_planner, "mkm", dt, 1, Ps, Ps, opX=capi.OP_T)
        assert e == capi.SUCCESS and names == plain[1] and launches[0]["in"] == plain[2][0]["in"], (dt, Ps, names)


def test_the_pair_behind_a_copy_is_judged_by_its_merged_factors(online_planner):
    """Us without the copy / with it: 10.7 / 14.8, 10.7 / 13.8, 10.4 / 12.0."""
    for dt, M, Ps in [("s", 1673, [2] * 5), ("d", 213, [4] * 4), ("d", 548, [4] * 3)]:
        e, names, _ = plan(online_planner, "mkm", dt, M, Ps, Ps, opX=capi.OP_T)
        assert e == capi.SUCCESS and not any(n.startswith("transpose_") for n in names), (dt, M, Ps, names)


# ---- records and caches of a handle ----
@pytest.mark.parametrize("dt,M,P,N,key,steps", [("s", 88, 7, 4, "(7x7^4)*2401x88_NN_f", 4), ("d", 88, 7, 4, "(7x7^4)*2401x88_NN_d", 4),
                                                ("d", 1000, 4, 5, "(4x4(x)16x16(x)16x16)*1024x1000_NN_d", 3)])
def test_records_without_rewriting_fields_come_before_the_rules_for_columns(online_planner, tmp_path, dt, M, P, N, key, steps):
    """Plan files written before records said how a chain is rewritten hold it as the rules rewrote it (the last one: merged)."""
    lib, h = online_planner
    e, names, _ = plan(online_planner, "kmm", dt, M, [P] * N, [P] * N)
    assert e == capi.SUCCESS and any("columns" in n for n in names), names
    generic = "gekmm_hip_gfx950_256_%s_generic_1" % ("f" if dt == "s" else "d")
    f = tmp_path / "open.db"
    f.write_text(f"{key} 0.01 {steps} " + " ".join(f"{i} {i} {generic}" for i in reversed(range(steps))) + "\n")
    lib.fastKronSetTunedDB(h, str(f).encode())
    e, names, _ = plan(online_planner, "kmm", dt, M, [P] * N, [P] * N)
    assert e == capi.SUCCESS and names == [generic] * steps, names


COLUMNS = "kmm_hip_gfx950_512_%s_small_fused_columns_8"


@pytest.mark.parametrize("dt", ["s", "d"])
def test_records_of_groups_in_place_run_those_groups(online_planner, tmp_path, dt):
    """M2: the steps as problems on the columns behind them; records that do not fit a call leave it to the rules."""
    lib, h = online_planner
    k, t = COLUMNS % ("f" if dt == "s" else "d"), "f" if dt == "s" else "d"
    key = "(7x7^5)*16807x5_NN_" + t
    other = plan(online_planner, "kmm", dt, 5, [7] * 5, [7] * 5)[1]
    f = tmp_path / "groups.db"
    def run(line, **kw):
        f.write_text(line + "\n")
        lib.fastKronSetTunedDB(h, str(f).encode())
        e, names, launches = plan(online_planner, "kmm", dt, 5, [7] * 5, [7] * 5, **kw)
        assert e == capi.SUCCESS
        return names, [(int(l["M"]), int(l["batch"])) for l in launches]
    # other groups than the rule's (2 and 3 factors), so that the record is what runs
    assert run(f"{key} 0.01 M2 S0 2 2 4 {k} 0 1 {k}") == ([k] * 2, [(5, 49), (5 * 343, 1)])
    assert run(f"{key} 0.01 M2 S0 2 3 4 {k} 0 2 {k}") == ([k] * 2, [(5, 343), (5 * 49, 1)])
    for bad in ("2 0 1 %s 2 4 %s" % (k, k), "2 2 4 %s 1 1 %s" % (k, k), "1 2 4 %s" % k, "2 1 4 %s 0 0 %s" % (k, k), "2 2 4 nothing 0 1 %s" % k):
        assert run(f"{key} 0.01 M2 S0 {bad}")[0] == other, bad
    # one temporary holds what two launches pass on; factors of each entry's own and gaps in X rule the groups out
    assert run(f"{key} 0.01 M2 S0 2 2 4 {k} 0 1 {k}", temp2=False)[0] == [k] * 2
    batched = "(7x7^5)*16807x5_NN_%s_stridedBatched_2" % t
    assert run(f"{batched} 0.01 M2 S0 2 2 4 {k} 0 1 {k}", batch=2)[0] == plan(online_planner, "kmm", dt, 5, [7] * 5, [7] * 5, batch=2)[1]
    own, _ = run(f"{batched} 0.01 M2 S0 2 2 4 {k} 0 1 {k}", batch=2)
    assert k not in own
    gaps, _ = run(f"{batched}_Fs1f 0.01 M2 S0 2 2 4 {k} 0 1 {k}", batch=2, strideF=[0] * 5, strides={"x": 5 * 7 ** 5 + 8})
    assert k not in gaps
    assert run(f"{batched}_Fs1f 0.01 M2 S0 2 2 4 {k} 0 1 {k}", batch=2, strideF=[0] * 5)[1] == [(5, 98), (5 * 343, 2)]


def test_a_handle_keeps_a_bounded_number_of_plans(online_planner):
    """Calls with ever new row counts: what the handle remembers of them stops growing (50000 problems took 34 MB)."""
    import os
    lib, h = online_planner
    page = os.sysconf("SC_PAGE_SIZE")
    resident = lambda: int(open("/proc/self/statm").read().split()[1]) * page
    def calls(lo, hi):
        ps, x = capi.arr_u32([24] * 3), ctypes.c_void_p(BASE)
        fs = capi.arr_ptr([BASE] * 3)
        for M in range(lo, hi):
            assert lib.sgemkm(h, capi.BACKEND_HIP, M, 3, ps, ps, x, capi.OP_T, fs, capi.OP_N, x, ctypes.c_float(1), ctypes.c_float(0), None, x, x) == 0
    calls(1, 12000)
    before = resident()
    calls(12000, 62000)
    assert resident() - before < 8 << 20


def test_workgroups_that_go_from_tile_to_tile_make_no_second_round_for_a_few(tmp_path):
    """persistentWorkgroups (csrc/problem.h) on its own: as many per part as fit, or one more each where that ends earlier."""
    import os
    import subprocess
    src = tmp_path / "count.cpp"
    src.write_text("""
#include <cstdio>
#include "problem.h"
int main() {
  unsigned need, share, places;
  while (scanf("%u %u %u", &need, &share, &places) == 3) printf("%u\\n", fk::persistentWorkgroups(need, share, places));
}
""")
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fastkron_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-I", csrc, str(src), "-o", str(tmp_path / "count")], check=True)
    cases = [(need, share, places) for places in (256, 512, 1024) for share in (1, 2, 3, 5, 7, 12, 36, 255, 256, 300, 4000) for need in (1, 2, 9, 85, 86, 97, 927, 20000)]
    out = subprocess.run([str(tmp_path / "count")], input="\n".join("%d %d %d" % c for c in cases), capture_output=True, text=True, check=True).stdout
    up = lambda a, b: -(-a // b)
    for (need, share, places), w in zip(cases, map(int, out.split())):
        time = lambda n: up(n * share, places) * up(need, n)
        assert 1 <= w <= need and time(w) <= time(min(need, max(1, places // share))) and time(w) <= time(min(need, up(places, share))), (need, share, places, w)
    answer = dict(zip(cases, map(int, out.split())))
    assert answer[(927, 3, 256)] == 85 and answer[(20000, 7, 512)] == 73 and answer[(1, 1, 256)] == 1 and answer[(9, 1, 256)] == 9
