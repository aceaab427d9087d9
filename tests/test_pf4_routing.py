"""Which launch a prefill call takes (pick_pf16, pick_pf4 in csrc/qmm.hip): few
output tiles a CU go to independent 16-row waves (pf_rp 0), more to a
workgroup shape, for INT4 the one of least cost (kPf4Costs)."""
import pytest

TABLE = [
    # (M, K, N) -> plan fields
    ((33, 5120, 5120), dict(pf_rp=0, grid_x=240, grid_y=1)),
    ((64, 17408, 5120), dict(pf_rp=0, grid_x=320)),
    ((166, 4096, 4096), dict(pf_rp=0, grid_x=704)),   # 11 tiles a CU
    ((256, 4096, 4096), dict(pf_rp=2, pf_ct=8)),      # 16
    ((64, 5120, 17408), dict(pf_rp=2, pf_ct=8, grid_x=136, grid_y=1)),
    ((200, 5120, 17408), dict(pf_rp=4, pf_ct=9, grid_x=121, grid_y=2)),
    ((512, 5120, 17408), dict(pf_rp=4, pf_ct=17, grid_x=64, grid_y=4)),
]


@pytest.mark.parametrize("shape,want", TABLE, ids=[str(t[0]) for t in TABLE])
def test_int4_prefill_launch(hb, shape, want):
    M, K, N = shape
    got = hb.plan(4, M, K, N, n_cu=256)
    assert got["route"] == "prefill"
    assert {k: got[k] for k in want} == want, got


def test_overrides(hb, monkeypatch):
    monkeypatch.setenv("BREEZE_HIP_PF16", "0")
    assert hb.plan(4, 33, 5120, 5120)["pf_rp"] != 0
    monkeypatch.setenv("BREEZE_HIP_PF16", "1")
    assert hb.plan(4, 512, 5120, 17408)["pf_rp"] == 0
    monkeypatch.delenv("BREEZE_HIP_PF16")
    monkeypatch.setenv("BREEZE_HIP_PREFILL_RP", "2")
    monkeypatch.setenv("BREEZE_HIP_PREFILL_CT", "16")
    p = hb.plan(4, 33, 5120, 5120)
    assert (p["pf_rp"], p["pf_ct"]) == (2, 16)


@pytest.mark.parametrize("shape,want", [
    ((8, 64, 5120, 5120), dict(pf_rp=0, grid_x=320)),
    ((8, 48, 5120, 10240), dict(pf_rp=0, grid_x=480)),  # 7.5 tiles a CU
    # 12.75, where the waves were taken at first: with the weights in the
    # memory-side cache 57 us against 63 on workgroups, from memory 74 against 64.
    ((8, 48, 5120, 17408), dict(pf_rp=2)),
    ((8, 64, 5120, 17408), dict(pf_rp=2)),              # 17
    ((8, 512, 5120, 17408), dict(pf_rp=4, pf_ct=17)),
])
def test_int8_prefill_launch(hb, shape, want):
    got = hb.plan(*shape, n_cu=256)
    assert got["route"] == "prefill"
    assert {k: got[k] for k in want} == want, got


def test_int8_waves_that_are_faster_either_way(hb):
    """INT8 activations, K=1024 N=12288, 33 rows: waves 10.4 us with the weights
    in the memory-side cache and 11.9 from memory, workgroups 12.4 and 12.6;
    K=2048: 14.6 and 18.1, 19.1 and 19.5.  K=5120 N=12288 with per-block scales,
    where the waves lose 15% from memory, stays on workgroups."""
    for K in (1024, 2048):
        for M in (33, 48, 64):
            assert hb.plan(8, M, K, 12288, hi=False)["pf_rp"] == 0
    assert hb.plan(8, 33, 5120, 12288, hi=False, extra=True)["pf_rp"] == 2


def test_projections_share_a_prefill_launch(hb):
    """Past 32 rows the gate/up pair (twice the tiles) and multi-projection
    calls take one INT4 prefill launch; INT8 ones, the fused norm, argmax and
    a legacy corr do not."""
    p = hb.plan(4, 200, 5120, 17408, pair=True)
    assert (p["route"], p["pf_rp"], p["pf_ct"], p["grid_x"], p["grid_y"]) == ("prefill", 4, 17, 128, 2)
    assert hb.plan(4, 64, 5120, 10240, multi=True)["route"] == "prefill"
    assert hb.plan(4, 64, 5120, 10240, multi=True, extra=True)["route"] == "prefill"
    assert hb.plan(4, 32, 4096, 4096, pair=True)["route"] is None
    assert hb.plan(8, 64, 5120, 10240, multi=True)["route"] is None
    assert hb.plan(4, 64, 5120, 10240, multi=True, norm=True)["route"] is None
    assert hb.plan(4, 64, 5120, 10240, multi=True, argmax=True)["route"] is None
    assert hb.plan(4, 64, 5120, 10240, pair=True, legacy_corr=True)["route"] is None


@pytest.mark.parametrize("M", [33, 64, 100, 128, 256, 512, 1000, 4096])
@pytest.mark.parametrize("N", [16, 48, 1024, 5120, 17408, 151936])
def test_every_output_is_covered(hb, M, N):
    p = hb.plan(4, M, 5120, N)
    if p["route"] != "prefill":
        return
    if p["pf_rp"] == 0:
        assert p["grid_x"] * 4 >= N // 16 * -(-M // 16)
    else:
        assert p["grid_x"] * p["pf_ct"] >= N // 16 and p["grid_y"] * 32 * p["pf_rp"] >= M


@pytest.mark.parametrize("M,N", [(33, 5120), (128, 17408)])
def test_zero_points_are_read_only_where_given(hb, M, N):
    """Per-block scales alone (extra) leave the zero points at 8: the kernels
    without them.  INT8 weights have none."""
    assert hb.plan(4, M, 5120, N)["pf_zp"] == 0
    assert hb.plan(4, M, 5120, N, extra=True)["pf_zp"] == 0
    assert hb.plan(4, M, 5120, N, zeros=True)["pf_zp"] == 1
    assert hb.plan(4, M, 5120, N, pair=True, zeros=True)["pf_zp"] == 1
    assert hb.plan(8, M, 5120, N, extra=True)["pf_zp"] == 0


COSTS = [
    # (M, K, N), call -> (row pairs, column tiles) of the launch; zeros: explicit
    # zero points, hi: two-pass activations.  Five tiles a workgroup where they
    # fill one round that eight would leave half empty, whatever K and the mode.
    ((128, 5120, 17408), dict(), (4, 5)),
    ((128, 5120, 17408), dict(zeros=True), (4, 5)),
    ((128, 5120, 17408), dict(zeros=True, hi=False), (4, 5)),
    ((100, 5120, 17408), dict(zeros=True), (4, 5)),
    ((128, 1024, 17408), dict(), (4, 5)),
    ((128, 2048, 17408), dict(zeros=True), (4, 5)),
    ((400, 5120, 5120), dict(zeros=True), (4, 5)),
    ((200, 5120, 10240), dict(zeros=True), (4, 5)),
    # 12.5 output tiles a CU: independent waves only without zero points, two
    # passes, where the bound of 13 stands.
    ((320, 5120, 2560), dict(), (0, 1)),
    ((320, 5120, 2560), dict(zeros=True, hi=False), (2, 4)),
    ((160, 2048, 5120), dict(zeros=True, hi=False), (2, 4)),
    # Fewer: independent waves in every mode.
    ((64, 5120, 5120), dict(zeros=True), (0, 1)),
    ((64, 5120, 5120), dict(hi=False), (0, 1)),
    # The largest shapes are those that fill one round.
    ((512, 5120, 17408), dict(zeros=True, hi=False), (4, 17)),
    ((200, 5120, 17408), dict(zeros=True), (4, 9)),
]


@pytest.mark.parametrize("shape,call,want", COSTS, ids=[f"{c[0]}{c[1]}" for c in COSTS])
def test_int4_launch_of_least_cost(hb, shape, call, want):
    p = hb.plan(4, *shape, n_cu=256, **call)
    assert (p["pf_rp"], p["pf_ct"]) == want, p


@pytest.mark.parametrize("call", [dict(zeros=True), dict(hi=False), dict(zeros=True, hi=False),
                                  dict(pair=True, zeros=True, hi=False)])
@pytest.mark.parametrize("M", [33, 100, 320, 1000])
@pytest.mark.parametrize("N", [16, 48, 2560, 17408, 27648])
def test_every_output_is_covered_in_every_mode(hb, M, N, call):
    p = hb.plan(4, M, 1024, N, **call)
    tiles = N // 16 * (2 if call.get("pair") else 1)
    if p["pf_rp"] == 0:
        assert p["grid_x"] * 4 >= tiles * -(-M // 16)
    else:
        assert p["grid_x"] * p["pf_ct"] >= tiles and p["grid_y"] * 32 * p["pf_rp"] >= M


def test_zero_points_under_int8_activations(hb, monkeypatch):
    """One projection past 64 rows with explicit zero points, INT8 activations:
    the INT8 instructions where their cost is less."""
    call = dict(zeros=True, hi=False)
    assert hb.plan(4, 128, 5120, 17408, **call)["pf_i8"] == 1
    assert hb.plan(4, 400, 1024, 5120, **call)["pf_i8"] == 1
    assert hb.plan(4, 1024, 2048, 17408, **call)["pf_i8"] == 1
    assert hb.plan(4, 320, 5120, 2560, **call)["pf_i8"] == 0    # FP6, (2, 4)
    assert hb.plan(4, 96, 5120, 5120, **call)["pf_rp"] == 0     # independent waves
    assert hb.plan(4, 64, 5120, 17408, **call)["pf_i8"] == 0
    assert hb.plan(4, 128, 5120, 17408, pair=True, **call)["pf_i8"] == 0
    assert hb.plan(4, 128, 5120, 17408, hi=False, extra=True)["pf_i8"] == 0
    assert hb.plan(4, 128, 5120, 17408, zeros=True)["pf_i8"] == 0
    assert hb.plan(8, 128, 5120, 17408, hi=False)["pf_i8"] == 0
    monkeypatch.setenv("BREEZE_HIP_PF_I8", "0")
    assert hb.plan(4, 128, 5120, 17408, **call)["pf_i8"] == 0
    monkeypatch.setenv("BREEZE_HIP_PF_I8", "1")
    assert hb.plan(4, 64, 5120, 17408, **call)["pf_i8"] == 1


@pytest.mark.parametrize("shape,call,waves", [
    ((64, 5120, 5120), dict(), True),
    ((64, 5120, 5120), dict(extra=True), True),
    ((64, 5120, 5120), dict(hi=False, extra=True), True),
    ((128, 5120, 5120), dict(), True),
    ((48, 5120, 17408), dict(extra=True), False),   # four workgroups on the busiest CU
    ((17, 5120, 17408), dict(), False),
    ((64, 12288, 10240), dict(), False),
    ((48, 5120, 10240), dict(hi=False), True),
    ((80, 5120, 10240), dict(extra=True), False),
    ((24, 12288, 17408), dict(extra=True), False),
    ((33, 1024, 17408), dict(extra=True), False),
    ((320, 5120, 2560), dict(extra=True), False),
])
def test_int8_waves_where_they_cost_less(hb, shape, call, waves):
    """Per-block scales make the independent waves' step longer, INT8
    activations shorter; workgroups change little."""
    assert (hb.plan(8, *shape, n_cu=256, **call)["pf_rp"] == 0) == waves


def test_weight_chunks_in_flight(hb, monkeypatch):
    """Four up to six output tiles a CU, two past that."""
    assert hb.plan(4, 33, 5120, 5120)["pf_ahead"] == 4               # 960 waves
    assert hb.plan(4, 77, 5120, 5120, zeros=True, hi=False)["pf_ahead"] == 2  # 1600
    assert hb.plan(4, 166, 4096, 4096)["pf_ahead"] == 2              # 2816
    monkeypatch.setenv("BREEZE_HIP_PF16_AHEAD", "2")
    assert hb.plan(4, 33, 5120, 5120)["pf_ahead"] == 2


@pytest.mark.parametrize("zeros", [False, True])
def test_every_shape_can_be_forced(hb, monkeypatch, zeros):
    for rp, cts in ((4, (17, 16, 13, 12, 9, 8, 5, 4)), (2, (16, 8, 4)), (1, (16, 8))):
        monkeypatch.setenv("BREEZE_HIP_PREFILL_RP", str(rp))
        for ct in cts:
            monkeypatch.setenv("BREEZE_HIP_PREFILL_CT", str(ct))
            p = hb.plan(4, 130, 1056, 304, zeros=zeros)
            assert (p["pf_rp"], p["pf_ct"]) == (rp, ct)
