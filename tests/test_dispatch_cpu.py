"""The scratch the library reserves for a MUL_MAT covers what the kernel launchers it picks ask for.

qproj_workspace_bytes walks the library's own dispatch (the code that serves qproj_mul_mat_multi) without
launching: every launcher works out its demand from the variables that pick its split and refuses a buffer that is
too small, so a sizing rule and a dispatch rule that disagree show up here, on the CPU, as a non-zero status --
not as a write past a device buffer."""
import itertools
import re

import pytest

from magnitude_amd import qproj

Q8_0, Q4_K, Q6_K = 8, 12, 14
GGML, F32, Q8X32 = 0, 1, 2

MS = [1, 2, 3, 4, 5, 8, 9, 15, 16, 17, 20, 31, 32, 33, 47, 48, 63, 64, 65, 96, 127, 128, 129, 200, 255, 256, 333, 511, 512,
      513, 1000, 1024, 2048, 4096]
KS = [256, 512, 768, 1024, 2048, 3072, 4096, 5120, 6144, 8192, 11008, 14336, 28672]
NS = [(1,), (5,), (32,), (77,), (128,), (256,), (1024,), (4096,), (14336,), (4096, 1024, 1024), (14336, 14336), (768, 768),
      (130, 5), (1024, 1024, 1024, 1024), (32000,)]


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K, Q8_0])
def test_every_launcher_is_satisfied_by_the_reserved_scratch(qtype):
    checked = 0
    for m, k, ns in itertools.product(MS, KS, NS):
        nbytes = qproj.workspace_bytes(qtype, k, ns, m, GGML)       # raises on a launcher that would be refused
        if m <= 2 or (m <= 4 and (k <= 4096 or (qtype == Q8_0 and k <= 20480))):   # (four Q8_0 rows of K <= 20480 fit the kernel's LDS)
            assert nbytes == 0, (m, k, ns)                            # decode regime: the kernel quantizes its own rows
        else:
            assert nbytes >= qproj.load_library().qproj_act_bytes(GGML, qtype, m, k) > 0
        checked += 1
    assert checked == len(MS) * len(KS) * len(NS)


def test_q8_0_rows_of_whole_blocks_only():
    for m, k in itertools.product([1, 3, 16, 17, 64, 100, 512], [32, 96, 288, 1056, 4096 + 32]):
        qproj.workspace_bytes(Q8_0, k, (77,), m, GGML)


def test_per32_and_fp32_modes():
    for m, k, ns in itertools.product([1, 3, 17, 64, 200, 512, 2048], [256, 4096, 14336], [(4096,), (14336,), (130,)]):
        nbytes = qproj.workspace_bytes(Q4_K, k, ns, m, Q8X32)
        assert nbytes >= qproj.load_library().qproj_act_bytes(Q8X32, Q4_K, m, k)
        assert qproj.workspace_bytes(Q4_K, k, ns, m, F32) == 0
    with pytest.raises(qproj.QprojError):
        qproj.workspace_bytes(Q6_K, 4096, (4096,), 64, Q8X32)        # the per-32 path is built for Q4_K weights


def test_known_sizes():
    al = lambda v: (v + 255) // 256 * 256
    planes = lambda m, k: al(m * k) + al(m * (k // 256) * 4) + al(m * (k // 16) * 2) + al(m * (k // 256) * 32) + al(m * 4)
    # down projection of the 8B layer at 512 tokens: 64 tiles of 128 tokens x 256 rows for 256 compute units, K is cut in four
    assert qproj.workspace_bytes(Q6_K, 14336, (4096,), 512, GGML) == planes(512, 14336) + 4 * 512 * 4096 * 4
    # gate/up at 4096 tokens: the grid is full, nothing beyond the activation planes
    assert qproj.workspace_bytes(Q4_K, 4096, (14336, 14336), 4096, GGML) == planes(4096, 4096)
    # small batch, K = 14336 at 16 rows: per-chunk results of the small-batch kernel
    assert qproj.workspace_bytes(Q6_K, 14336, (4096,), 16, GGML) > planes(16, 14336)


def test_bad_shapes_are_refused():
    lib = qproj.load_library()
    import ctypes as C
    st = C.c_int(0)
    arr = (C.c_int64 * 1)(4096)
    assert lib.qproj_workspace_bytes(Q4_K, 4100, 1, arr, 4, GGML, C.byref(st)) == 0 and st.value == 1
    assert lib.qproj_workspace_bytes(2, 4096, 1, arr, 4, GGML, C.byref(st)) == 0 and st.value == 1
    assert lib.qproj_workspace_bytes(Q4_K, 4096, 5, arr, 4, GGML, C.byref(st)) == 0 and st.value == 1
    assert lib.qproj_workspace_bytes(Q4_K, 4096, 1, None, 4, GGML, None) == 0


def test_the_8b_layer_fits_the_fixed_scratch_up_to_512_tokens():
    """The allocation-free entry point keeps its scratch in a fixed 64 MiB buffer: every projection group of the
    8B-class layer must fit for the batches the engine issues (n_batch 512,
    /root/reference/inference/crates/icn-engine/src/lib.rs:93-96)."""
    groups = [(Q4_K, 4096, (4096, 1024, 1024)), (Q4_K, 4096, (4096,)), (Q4_K, 4096, (14336, 14336)), (Q6_K, 14336, (4096,))]
    for m in (1, 2, 4, 8, 16, 64, 128, 512):
        for qt, k, ns in groups:
            assert qproj.workspace_bytes(qt, k, ns, m, GGML) <= qproj.NOALLOC_SCRATCH_BYTES, (m, qt, k, ns)
    assert qproj.workspace_bytes(Q6_K, 14336, (4096,), 4096, GGML) > qproj.NOALLOC_SCRATCH_BYTES   # and larger ones are refused


# ---------------------------------------------------------------------------------------------------------------
# The routing table: which kernel, tile, grid and cuts of K serve every shape of the benchmark configurations.  The
# lines are written by the launchers themselves in a dry run of the dispatch (qproj_plan_mul_mat / qproj_plan_moe_ffn),
# so an edit of a routing threshold shows up as a diff of tests/golden/dispatch_plan.txt.
# Regenerate after a deliberate change with:  QPROJ_UPDATE_PLAN=1 python -m pytest tests/test_dispatch_cpu.py -k routing_table
def routing_table() -> str:
    out = []

    def dense(title, qtype, k, ns, m, act=GGML, with_norm=False):
        out.append(f"## {title}: {'Q8_0' if qtype == Q8_0 else 'Q4_K' if qtype == Q4_K else 'Q6_K'} K={k} N={list(ns)} M={m} "
                   f"act={'ggml' if act == GGML else 'f32' if act == F32 else 'q8x32'}{' +rms_norm' if with_norm else ''}")
        out.append(qproj.plan_mul_mat(qtype, k, ns, m, act, with_norm).rstrip())

    layer = [("q/k/v", Q4_K, 4096, (4096, 1024, 1024)), ("o", Q4_K, 4096, (4096,)), ("gate/up", Q4_K, 4096, (14336, 14336)),
             ("down", Q6_K, 14336, (4096,))]
    dense("config 1", Q8_0, 4096, (4096,), 1)
    for name, qt, k, ns in layer:
        dense(f"config 2 {name}", qt, k, ns, 1)
    dense("config 2 norm + q/k/v", Q4_K, 4096, (4096, 1024, 1024), 1, with_norm=True)
    dense("config 2 norm + gate/up", Q4_K, 4096, (14336, 14336), 1, with_norm=True)
    for m in (2, 4, 8, 16):
        for name, qt, k, ns in layer:
            dense(f"config 3 {name}", qt, k, ns, m)
    for m in (512, 2048, 4096):
        for k, n in ((4096, 14336), (14336, 4096), (4096, 4096)):
            dense("config 4 (per-32 activations)", Q4_K, k, (n,), m, Q8X32)
            dense("config 4 (ggml activations)", Q4_K, k, (n,), m)
        dense("config 4 (ggml activations) down", Q6_K, 14336, (4096,), m)
        dense("config 4 (ggml activations) config 1's matrix", Q8_0, 4096, (4096,), m)
    for name, qt, k, ns in layer:
        dense(f"prompt batch of the engine (512 tokens) {name}", qt, k, ns, 512)
    # batches of 33..256 rows: streamed K-quants (one matrix alone, both workgroup sizes), shared Q8_0 launches
    for m in (48, 96, 128, 187, 256):
        for name, qt, k, ns in layer:
            dense(f"serving batch {name}", qt, k, ns, m)
    for m in (48, 187, 256):
        dense("serving batch gate alone", Q4_K, 4096, (14336,), m)
        dense("serving batch, Q6_K q/k/v", Q6_K, 4096, (4096, 1024, 1024), m)
        dense("serving batch, Q6_K gate/up", Q6_K, 4096, (14336, 14336), m)
        dense("serving batch, output head", Q6_K, 4096, (32000,), m)
        dense("serving batch, long rows", Q6_K, 8192, (8192, 1024, 1024), m)
        dense("serving batch, long rows", Q4_K, 28672, (8192,), m)
        for name, k, ns in (("q/k/v", 3072, (3072, 1024, 1024)), ("o", 3072, (3072,)), ("gate/up", 3072, (8192, 8192)), ("down", 8192, (3072,))):
            dense(f"serving batch, Q8_0 {name}", Q8_0, k, ns, m)
    for b in (1, 8, 64, 500):
        out.append(f"## config 5: 128 experts, top-8, d_model 2048, d_ff 768, Q4_K, B={b}")
        out.append(qproj.plan_moe_ffn(Q4_K, Q4_K, 2048, 768, 128, 8, b).rstrip())
    return "\n".join(out) + "\n"


def test_routing_table_of_the_benchmark_configurations_is_pinned():
    import os
    path = os.path.join(os.path.dirname(__file__), "golden", "dispatch_plan.txt")
    table = routing_table()
    if os.environ.get("QPROJ_UPDATE_PLAN"):
        with open(path, "w") as f:
            f.write(table)
    with open(path) as f:
        pinned = f.read()
    assert table == pinned, "the dispatch changed: review the diff, then regenerate tests/golden/dispatch_plan.txt"
    # every shape is served (no refusal) and the decode regime stays one launch
    assert "refused" not in table
    first = table.split("## config 2 q/k/v")[1].split("##")[0]
    assert first.count("gemv_decode_kernel") == 1 and "quantizer:" not in first


def test_plan_names_kernels_that_are_launched():
    """A line of the plan is matched to a profile by the kernel's name: every name is one that the sources define, and the small
    batches, whose products have a dense and an expert-grouped kernel, name the one they launch."""
    import glob
    import os
    sources = "".join(open(f).read() for f in glob.glob(os.path.join(os.path.dirname(qproj.__file__), "csrc", "*.hip")))
    defined = set(re.findall(r"__global__[^;{]*?void\s+(\w+)\s*\(", sources))
    plans = [routing_table()] + [qproj.plan_mul_mat(qt, 4096, (4096,), m) for qt in (Q8_0, Q4_K, Q6_K) for m in (5, 8, 16, 32)]
    named = set(re.findall(r"\b(\w+_kernel\w*)\b", "".join(plans)))
    assert named <= defined, named - defined
    for plan in plans[1:]:
        assert "gemv_mfma_dense_kernel<" in plan and "gemv_mfma_kernel<" not in plan, plan
    grouped = qproj.plan_moe_ffn(Q6_K, Q6_K, 2048, 768, 128, 8, 64)
    assert grouped.count("gemv_mfma_kernel<") == 2 and "dense" not in grouped, grouped


@pytest.mark.parametrize("k,parts", [(32, 2), (1024, 2), (2048, 2), (2080, 3), (3072, 3), (3104, 4), (4096, 4), (4128, 3), (5120, 3), (6144, 3),
                                     (6176, 4), (8192, 4), (8224, 3), (9216, 3), (9248, 4), (12288, 4), (12320, 4), (13824, 4), (14336, 4),
                                     (15360, 4), (16896, 4), (18432, 4)])
def test_q8_0_decode_steps_take_three_parts_where_a_quarter_fewer_are_needed(k, parts):
    """Two parts of 1024 weights a step for rows that they cover, three where steps of four would take a third more, for one to
    four activation rows.  Longer rows than nine parts keep four: their sums are further from 64 bits in steps of three."""
    for m in (1, 2, 4):
        plan = qproj.plan_mul_mat(Q8_0, k, (512, 512), m)
        assert re.findall(r"gemv_decode_kernel<Q8_0, (\d) parts of 1024 weights a step,", plan) == [str(parts)], plan
    assert "gemv_decode_kernel<Q4_K, 1 activation rows" in qproj.plan_mul_mat(Q4_K, k // 256 * 256 + 256, (512,), 1)


def test_plan_reports_a_refused_call():
    with pytest.raises(qproj.QprojError):
        qproj.plan_mul_mat(Q6_K, 4096, (4096,), 64, Q8X32)


def test_q8_0_matrices_share_a_launch_only_while_their_partial_results_have_room():
    # 256 rows of K = 196608: the activation planes leave 10 MB of the allocation-free entry point's 64 MiB, one matrix's
    # partial results are 4 MB, four matrices' 16
    k, ns = 196608, [1024] * 4
    plan = qproj.plan_mul_mat(Q8_0, k, ns, 256)
    assert plan.count("gemm_per32_kernel") == 4 and "(same launch)" not in plan
    assert 0 < qproj.workspace_bytes(Q8_0, k, ns, 256) <= 64 << 20
    assert qproj.plan_mul_mat(Q8_0, k // 2, ns, 256).count("(same launch)") == 3


@pytest.mark.parametrize("qtype,m", [(Q4_K, 64), (Q6_K, 48), (Q6_K, 96), (Q6_K, 192)])
def test_outputs_beyond_32_bit_indices_stay_on_the_kernels_with_64_bit_ones(qtype, m):
    """The streaming kernel indexes a tile's outputs with 32 bits (127 rows * N + 31 at most): matrices beyond 2^24 rows
    take the tiled kernels, whose output index has 64."""
    assert "gemm_stream_kernel" in qproj.plan_mul_mat(qtype, 256, [1 << 24], m)
    for n in ((1 << 24) + 1, 33_800_000, 40_000_000, 1 << 30):
        plan = qproj.plan_mul_mat(qtype, 256, [n], m)
        assert "gemm_stream_kernel" not in plan and "q8k" in plan, plan


@pytest.mark.parametrize("qtype", [Q4_K, Q6_K])
def test_streamed_batches_fit_the_fixed_scratch_while_their_activation_planes_do(qtype):
    """The partial tiles of a streamed call share what the 64 MiB of the allocation-free entry point leave beside the
    activation planes: one matrix's K is cut in no more stretches than fit there, and matrices whose partial tiles do
    not fit side by side go one after the other through the same bytes."""
    lib = qproj.load_library()
    apart = checked = 0
    for k, m in itertools.product([4096, 8192, 14336, 16384, 28672, 65536, 131072, 163840, 196608], [33, 64, 65, 96, 128, 187, 250, 256]):
        planes = lib.qproj_act_bytes(GGML, qtype, m, k)
        for ns in [(1024,), (8192,), (77,), (128,), (512,), (8192, 8192), (8192, 1024, 1024), (4096, 4096), (4096,) * 4, (512,) * 4, (28672, 28672)]:
            plan = qproj.plan_mul_mat(qtype, k, ns, m)
            if plan.count("gemm_stream_kernel") < len(ns):
                continue
            checked += 1
            nbytes = qproj.workspace_bytes(qtype, k, ns, m)
            assert planes <= nbytes <= max(planes, qproj.NOALLOC_SCRATCH_BYTES), (k, m, ns, nbytes)
            apart += plan.count("(same launch)") < len(ns) - 1
    assert checked > 300 and apart > 10
    assert qproj.workspace_bytes(Q6_K, 8192, (8192, 1024, 1024), 256) <= qproj.NOALLOC_SCRATCH_BYTES
    assert "(same launch)" in qproj.plan_mul_mat(Q6_K, 8192, (8192, 1024, 1024), 128)   # with room: one launch


@pytest.mark.parametrize("qtype", [Q8_0, Q4_K, Q6_K])
def test_a_matrix_is_cut_the_same_way_alone_and_beside_others(qtype):
    """Tile and stretches of K decide the order of a result's fp32 sums.  Q8_0 tiles and the streaming kernel take both
    from the matrix and the row count alone, so a call with several matrices gives the bits of separate calls."""
    def cuts(ns, k, m):   # kernel, tokens a tile, K parts, K stretches (how many rows a workgroup takes may follow the launch)
        lines = [l for l in qproj.plan_mul_mat(qtype, k, ns, m).splitlines() if "gemm_" in l]
        return [re.sub(r" x \d+ rows, \d+ tiles", "", l.replace(" (same launch)", "")) for l in lines]

    checked = 0
    for k, m in itertools.product([512, 3072, 4096, 8192, 14336], [33, 64, 100, 187, 256, 500, 2048]):
        for ns in [(4096, 1024, 1024), (8192, 8192), (3072, 1024, 1024), (28672, 28672), (512, 77, 2048, 256)]:
            together, alone = cuts(ns, k, m), [cuts((n,), k, m) for n in ns]
            if qtype != Q8_0 and any("gemm_stream_kernel" not in a[0] for a in alone):
                continue
            assert sorted(together) == sorted(sum(alone, [])), (k, m, ns)
            checked += 1
    assert checked > 30


def test_streamed_launches_that_would_fill_half_the_chip_take_half_the_rows_a_workgroup():
    for qtype, k, ns, m, rows in [(Q4_K, 4096, (14336,), 48, 64), (Q4_K, 4096, (14336, 14336), 48, 128), (Q6_K, 4096, (14336,), 160, 128),
                                  (Q6_K, 4096, (14336, 14336), 160, 256), (Q4_K, 4096, (32000,), 96, 128)]:
        plan = qproj.plan_mul_mat(qtype, k, ns, m)
        assert plan.count(f"x {rows} rows") == len(ns), plan


@pytest.mark.parametrize("qtype,d,tokens,first", [(Q4_K, 2048, 500, 32), (Q4_K, 2048, 640, 32), (Q4_K, 2048, 1000, 64), (Q4_K, 4096, 640, 48),
                                                  (Q6_K, 2048, 640, 48), (Q6_K, 2048, 360, 32), (Q6_K, 2048, 300, 16), (Q4_K, 2048, 64, 8),
                                                  (Q4_K, 2048, 160, 16)])
def test_experts_that_start_first_are_those_with_a_pass_more_than_the_average(qtype, d, tokens, first):
    """The line is a multiple of the rows a pass of the grouped launch stages: 32 only for Q4_K experts of up to 2048 weights
    a row with more than 16 pairs on average, 16 for the others, 8 up to four pairs."""
    plan = qproj.plan_moe_ffn(qtype, qtype, d, 768, 128, 8, tokens)
    assert f"those with more than {first} first" in plan, plan


def test_no_q8_0_stretch_of_k_is_empty():
    for k, n, m in itertools.product(range(512, 6144, 128), (1024, 3072, 8192), (64, 187, 500)):
        line = [l for l in qproj.plan_mul_mat(Q8_0, k, (n,), m).splitlines() if "gemm_per32_kernel" in l][0]
        stretches, units = int(re.search(r"x (\d+) K stretches", line)[1]), (k + 255) // 256
        assert (stretches - 1) * -(-units // stretches) < units, (k, n, m, line)


@pytest.mark.parametrize("cus", [16, 32, 38, 64, 76, 128, 152, 256, 304])
def test_every_call_is_served_whatever_the_number_of_compute_units(cus):
    """A partition of the GPU has fewer compute units (32 and 64 in its smaller modes), and the plans follow their number:
    what they name has to be there, and what a GPU of 256 units serves is served on the others."""
    lib = qproj.load_library()
    lib.qproj_internal_plan_cus(cus)
    try:
        for qt, m, k, ns in itertools.product([Q8_0, Q4_K, Q6_K], [3, 16, 33, 48, 64, 65, 96, 128, 129, 187, 192, 250, 300, 512, 2048],
                                              [512, 1536, 2048, 3072, 4096, 8192, 28672],
                                              [(512,), (1024,), (4096,), (6144,), (20480,), (32000,), (32768,), (4096, 1024, 1024), (8192, 8192), (3072, 3072, 3072)]):
            qproj.workspace_bytes(qt, k, ns, m)     # (raises where a launcher refuses)
        for tokens, experts, d, ff in itertools.product([1, 16, 64, 300], [8, 64, 256], [1024, 4096], [768, 2048]):
            qproj.plan_moe_ffn(Q4_K, Q4_K, d, ff, experts, 4, tokens)
    finally:
        lib.qproj_internal_plan_cus(0)


@pytest.mark.parametrize("m,k,ns", [(97, 2560, (2560, 1024, 1024)), (193, 3072, (3072, 1024, 1024)), (80, 2048, (2048, 2048, 2048)),
                                    (187, 3072, (1024,)), (48, 4096, (1024,))])
def test_q8_0_tiles_of_32_tokens_are_half_a_compute_unit(m, k, ns):
    """Workgroups of four waves: q/k/v beyond one round of larger ones would take two, and k or v alone would leave most of
    the chip idle."""
    plan = qproj.plan_mul_mat(Q8_0, k, ns, m)
    assert plan.count("gemm_per32_kernel_q8_0<1 token tiles") == plan.count("tile 32 tokens x 64 rows") == len(ns), plan


def q8_0_launch_workgroups(k, ns, m):
    """workgroups a launch of 96- or 64-token tiles with two K parts puts on the 8 XCDs (one a compute unit), 0 for other kernels"""
    lines = re.findall(r"gemm_per32_kernel_q8_0<[23] token tiles, 2 K parts>.* (\d+) tiles x (\d+) K stretches", qproj.plan_mul_mat(Q8_0, k, ns, m))
    return sum((int(tiles) + 7) // 8 * 8 * int(stretches) for tiles, stretches in lines)


def test_q8_0_stretches_are_one_round_on_every_xcd():
    """The stretches of a matrix are counted in workgroups as the XCDs get them: 36 tiles are five on four of them, so seven
    stretches are 35 workgroups for 32 compute units there."""
    seen = 0
    for k, n, m in itertools.product(range(1536, 16384, 512), range(1280, 8192, 256), (33, 64, 96, 129, 192)):
        if k > n:
            wgs = q8_0_launch_workgroups(k, (n,), m)
            assert wgs <= 256, (k, n, m, wgs)
            seen += wgs > 0
    assert seen > 500


def test_q8_0_gate_and_up_in_token_tiles_are_one_round_or_whole():
    """Cut in two so that its sums are no longer than those of the 128-token tiles, a gate / up pair of one round would be two."""
    seen = 0
    for k, f, m in itertools.product(range(1280, 4096, 256), (2.5, 3, 3.5, 4), (129, 160, 192)):
        n = 256 * round(k * f / 256)
        wgs = q8_0_launch_workgroups(k, (n, n), m)
        assert wgs <= 256, (k, n, m, wgs)
        seen += wgs > 0
    assert seen > 20


@pytest.mark.parametrize("m,k,n,stretches", [(160, 3072, 1536, 4), (129, 4096, 1280, 6), (80, 4096, 3072, 4), (96, 8192, 4096, 4), (192, 2560, 2304, 3)])
def test_q8_0_short_stretches_are_walked_in_halves_of_the_rows(m, k, n, stretches):
    """Eight waves and two to four steps of K a workgroup are mostly the start of a pipeline: half the rows and about half the
    stretches instead, never fewer than the 128-token tiles would make."""
    plan = qproj.plan_mul_mat(Q8_0, k, (n,), m)
    assert f"x 64 rows, {-(-m // 96) * (n // 64)} tiles x {stretches} K stretches of two levels of sums" in plan, plan


@pytest.mark.parametrize("m,k,n,rows", [(160, 6144, 3072, 128), (160, 14336, 4096, 128), (64, 4096, 3072, 128), (96, 5120, 1792, 64), (80, 5120, 1536, 64)])
def test_q8_0_longer_stretches_and_those_of_one_round_keep_one_level(m, k, n, rows):
    plan = qproj.plan_mul_mat(Q8_0, k, (n,), m)
    assert f"x {rows} rows" in plan and "two levels" not in plan, plan


@pytest.mark.parametrize("d,resident", [(2048, 2), (4096, 2), (7936, 2), (8192, 1)])
def test_expert_tiles_leave_room_for_a_second_workgroup(d, resident):
    """Two workgroups a compute unit, each filling the other's waits, but for the longest rows; the row tiles a workgroup walks are
    chosen by it."""
    plan = qproj.plan_moe_ffn(Q4_K, Q4_K, d, 1024, 128, 8, 64)
    gate = [l for l in plan.splitlines() if "moe_stream_kernel<Q4_K, gate" in l]
    assert len(gate) == 1 and gate[0].endswith(f"each, {resident} a compute unit"), plan


@pytest.mark.parametrize("experts,used,d,ff,tokens,tiles", [(128, 8, 2048, 2048, 56, False), (256, 8, 1024, 2048, 112, False), (64, 8, 4096, 2048, 28, False),
                                                            (16, 4, 4096, 2048, 16, False), (16, 4, 2048, 2048, 15, False), (16, 4, 4096, 2048, 17, True),
                                                            (128, 8, 2048, 768, 60, True), (32, 4, 4096, 1024, 32, True), (64, 8, 2048, 1024, 30, True)])
def test_expert_tiles_start_where_the_grouped_kernel_needs_second_passes(experts, used, d, ff, tokens, tiles):
    plan = qproj.plan_moe_ffn(Q4_K, Q4_K, d, ff, experts, used, tokens)
    assert plan.count("moe_stream_kernel") == (2 if tiles else 0), plan
