"""The small-tile kernel at the sizes where it can go wrong: edges of its row and column tiles, K
tails of a 128-deep step, each number of K groups, group sizes over 64, group scales that span more
than the int32 multipliers hold exactly, and output buffers that are not aligned to its stores.
Bar: bit-exact."""

import dataclasses

import numpy as np
import pytest

from oracle import qmm as oq
from qcom_htp_amd import cases as C

pytestmark = pytest.mark.gpu

# (M, K, N): one output block; row and column remainders with a K tail; 8 K groups with a tail; a
# row past a tile at many columns; a grid of wide tiles, for every width but 8 x 8 bits and for those
SHAPES = [(1, 32, 32), (33, 160, 96), (64, 1056, 1088), (65, 2048, 352), (700, 288, 2080), (700, 288, 4160)]
# ... requantised: the last four are the two K groups of the widest tiles and the GEMM just past them,
# for 16-bit and for 8-bit activations
REQUANT_SHAPES = [(17, 32, 32), (33, 160, 96), (65, 1184, 1088), (130, 4096, 480), (700, 288, 2080),
                  (330, 288, 2080), (500, 288, 2080), (700, 288, 4160), (1100, 288, 4160)]


def k_groups(cus, m, k, n, ab, cols, requant):
    """K groups of the kernel's workgroups (qmm_tile.hip, pick_split), cols channels per wave; 0: the
    GEMM's product (tile_pays)."""
    rows = 32 if ab == 16 else 64
    tiles = lambda ks: -(-m // rows) * -(-n // (cols * 8 // ks))  # noqa: E731
    if requant and tiles(2) > cus:
        return 0
    return 8 if -(-k // 128) >= 8 and tiles(8) <= cus else 4 if tiles(4) <= cus else 2


def test_shapes_reach_every_number_of_k_groups(gpu):
    import torch

    cus = torch.cuda.get_device_properties(gpu).multi_processor_count
    for ab in (8, 16):
        for wb in (8, 16):
            assert {k_groups(cus, *s, ab, 32 if wb == 16 else 64, False) for s in SHAPES} == {2, 4, 8}, (ab, wb)
        groups = [k_groups(cus, *s, ab, 32 if ab == 16 else 64, True) for s in REQUANT_SHAPES]
        assert set(groups) == {0, 2, 4, 8}, (ab, groups)


def unaligned(gpu, m, n, dtype):
    """A contiguous [m, n] buffer that starts one element past an allocation."""
    import torch

    return torch.empty(m * n + 1, dtype=dtype, device=gpu)[1:].view(m, n)


@pytest.mark.parametrize("mkn", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("bits", [(8, 8), (16, 8), (8, 16), (16, 16)], ids=lambda b: f"a{b[0]}w{b[1]}")
def test_contracts_and_accumulators(gpu, mkn, bits):
    import torch

    from qcom_htp_amd import _lib
    from qcom_htp_amd.qmm import QuantMatmul

    (m, k, n), (ab, wb) = mkn, bits
    rng = np.random.default_rng(m + k + n + ab)
    x = rng.integers(0, 1 << ab, size=(m, k)).astype(np.uint16 if ab == 16 else np.uint8)
    q = rng.integers(-32768 if wb == 16 else -127, 32768 if wb == 16 else 128, size=(n, k)).astype(np.int16)
    bias = rng.integers(-(1 << 20), 1 << 20, size=n).astype(np.int32)
    zp, out_zp = 3 << (ab - 3), 1 << (ab - 1)
    op = QuantMatmul(q if wb == 16 else q.astype(np.int8), np.ones(n, np.float32), bias, act_bits=ab, out_bits=ab,
                     act_scale=1.0, out_scale=1.0, act_zp=zp, out_zp=out_zp,
                     weight_format=_lib.QH_WEIGHT_I16 if wb == 16 else _lib.QH_WEIGHT_I8, device=gpu)
    act = torch.from_numpy(x).to(gpu)
    want = oq.int_accumulator(x, q, zp)
    np.testing.assert_array_equal(op.accumulate(act).cpu().numpy(), want)
    spread = max(1, int(np.abs(want).max()) >> (ab - 1))
    for name, d in (("clip_i32", 1), ("clip_i64", 1), ("div_rint", spread), ("div_rint", 2), ("floor256_div_rint", spread),
                    ("round_div", spread)):
        out = unaligned(gpu, m, n, op.out_dtype)
        got = op.run_contract(act, name, d, out=out).cpu().numpy()
        ref = oq.contract_output(want, name, d, bias, out_zp, ab)
        assert np.array_equal(got, ref), f"{name}/{d}: {(got != ref).sum()} differ"
    op.close()


@pytest.mark.parametrize("span", [0, 10], ids=["near_scales", "wide_scales"])
@pytest.mark.parametrize("mkng", [(1, 256, 32, 128), (33, 192, 96, 64), (64, 1280, 1088, 256), (65, 2048, 352, 1024),
                                  (700, 320, 2080, 64)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("fam", C.PER_GROUP_FAMILIES)
def test_per_group(gpu, fam, mkng, span):
    import torch

    from qcom_htp_amd.qmm import QuantMatmul

    m, k, n, gsz = mkng
    c = C.synthetic_case(fam, m, k, n, seed=m + k)
    rng = np.random.default_rng(k + n)
    s = rng.uniform(1e-3, 1e-2, size=(n, k // gsz)) * 2.0 ** rng.integers(-span, 1, size=(n, k // gsz))
    scale = s.astype(np.float32)
    deq = c.weight_q_nk.astype(np.float32) * np.repeat(scale, gsz, axis=1)
    x = (c.activation_q.astype(np.float64) - c.family.act_zp) * c.act_scale
    t = x @ deq.astype(np.float64).T + c.bias_float
    out_scale = C.affine_scale_from_minmax(float(t.min()), float(t.max()), 0, c.family.out_qmax, c.family.out_zp)
    c = dataclasses.replace(c, weight_scale=scale, weight_deq=deq, out_scale=out_scale)
    want = np.clip(np.rint(t / out_scale + c.family.out_zp), 0, c.family.out_qmax)
    op = QuantMatmul.from_case(c, device=gpu)
    got = op(torch.from_numpy(c.activation_q).to(gpu), out=unaligned(gpu, m, n, op.out_dtype)).cpu().numpy()
    op.close()
    assert np.array_equal(got, want.astype(got.dtype)), f"{(got != want).sum()} of {got.size} differ"


def per_group_8_to_16(m, k, n, gsz, span, coarse, tie, rng):
    """Operands of u8 activations, per-group int4 weights and u16 outputs; coarse: an output scale that
    uses a 2^-8 of the range; tie: odd dot products of the first rows on half-integers."""
    x = np.clip(np.rint(rng.normal(128.0, 40.0, size=(m, k))), 0, 255).astype(np.uint8)
    w = rng.integers(-7, 8, size=(n, k)).astype(np.int8)
    s = (rng.uniform(1e-3, 1e-2, size=(n, k // gsz)) * 2.0 ** rng.integers(-span, 1, size=(n, k // gsz))).astype(np.float32)
    sa, bias = 0.02, rng.uniform(-0.5, 0.5, size=n).astype(np.float32)
    if tie:
        sa, s = 2.0 ** -7, np.full_like(s, 2.0 ** -8)
        bias = (rng.integers(-8, 8, size=n) * (sa * 2.0 ** -8)).astype(np.float32)
        for r in range(min(m, 40)):
            x[r] = 128
            x[r, rng.choice(k, size=5, replace=False)] = 128 + rng.integers(-3, 4, size=5)
    t = ((x.astype(np.float64) - 128.0) * sa) @ (w.astype(np.float32) * np.repeat(s, gsz, axis=1)).astype(np.float64).T + bias
    so = 2.0 * sa * 2.0 ** -8 if tie else float(np.abs(t).max()) / 32767.0 * (256.0 if coarse else 1.0)
    return x, w, s, sa, bias, so, np.clip(np.rint(t / so + 32768.0), 0, 65535).astype(np.uint16)


def per_group_8_to_16_op(gpu, n, w, s, sa, bias, so, ob=16):
    from qcom_htp_amd import _lib
    from qcom_htp_amd.qmm import QuantMatmul

    return QuantMatmul(w, s, np.zeros(n, np.int32), act_bits=8, out_bits=ob, act_scale=sa, out_scale=so, act_zp=128,
                       out_zp=1 << (ob - 1), weight_format=_lib.QH_WEIGHT_I4_GROUP, bias_float=bias, device=gpu)


@pytest.mark.parametrize("span,coarse,tie", [(0, False, False), (10, False, False), (0, True, False), (0, False, True)],
                         ids=["fitted", "wide_scales", "coarse", "ties"])
@pytest.mark.parametrize("mkng", [(1, 256, 32, 128), (33, 192, 96, 64), (65, 2048, 352, 1024), (130, 4096, 480, 256),
                                  (700, 320, 2080, 64)], ids=lambda s: "x".join(map(str, s)))
def test_per_group_8_bit_to_16_bit(gpu, mkng, span, coarse, tie):
    """8-bit activations and 16-bit outputs, with the residue products (where many outputs would be
    uncertain without them) and without (a coarse output scale), at each number of K groups."""
    import torch

    m, k, n, gsz = mkng
    x, w, s, sa, bias, so, want = per_group_8_to_16(m, k, n, gsz, span, coarse, tie, np.random.default_rng(m + k))
    op = per_group_8_to_16_op(gpu, n, w, s, sa, bias, so)
    got = op(torch.from_numpy(x).to(gpu), out=unaligned(gpu, m, n, op.out_dtype)).cpu().numpy()
    op.close()
    assert np.array_equal(got, want), f"{(got != want).sum()} of {got.size} differ"


def test_per_group_16_bit_outputs_cost_little_more_than_8_bit_ones(gpu):
    """The time does not depend on how fine the output scale is: 12 against 10 us where recomputing every
    output that the left-out residues make uncertain took 65."""
    import torch

    m, k, n = 500, 2048, 2048
    x, w, s, sa, bias, so, _ = per_group_8_to_16(m, k, n, 64, 0, False, False, np.random.default_rng(1))
    act = torch.from_numpy(x).to(gpu)

    def best(ob):
        op = per_group_8_to_16_op(gpu, n, w, s, sa, bias, so * 2.0 ** (16 - ob), ob)
        times = []
        for _ in range(6):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(50):
                op(act)
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1) * 20.0)
        op.close()
        return min(times)

    t8, t16 = best(8), best(16)
    print(f"[tile] per-group {m}x{k}x{n}: u8 outputs {t8:.1f} us, u16 outputs {t16:.1f} us", flush=True)
    assert t16 <= 3.0 * t8


@pytest.mark.parametrize("ob", [8, 16], ids=["o8", "o16"])
@pytest.mark.parametrize("zp", ["low", "mid", "high"])
@pytest.mark.parametrize("ab,span", [(8, 20), (8, 25), (8, 28), (16, 14), (16, 17), (16, 20)], ids=lambda v: str(v))
def test_per_group_outputs_far_below_a_group_of_large_scale(gpu, ab, span, zp, ob):
    """Group scales 2^14 to 2^28 apart (the widest that prepare accepts), where the int32 multipliers round the small ones away, with the large
    group's activations at the zero point: the sums that the kernel forms are then off by many steps of
    the output, and each output whose error bound reaches the output range has to be recomputed, however
    far outside that range its sum lies."""
    import torch

    from qcom_htp_amd import _lib
    from qcom_htp_amd.qmm import QuantMatmul

    m, k, n = 70, 192, 96
    rng = np.random.default_rng(span + ab)
    azp = {"low": 0, "mid": 1 << (ab - 1), "high": (1 << ab) - 1}[zp]
    x = np.full((m, k), azp, dtype=np.int64)
    x[:, 64:128] = np.clip(azp + rng.integers(-30, 31, size=(m, 64)), 0, (1 << ab) - 1)
    w = rng.integers(-7, 8, size=(n, k)).astype(np.int8)
    w[: n // 2, :64] = 0
    w[: n // 2, 0] = 1  # one code in the large group; the other channels have 64 codes in one 2^-9 as large
    s = np.float32(rng.uniform(4e-3, 7e-3, size=(n, 3))) * np.float32([2.0 ** span, 1.0, 1.0])
    s[n // 2 :, 0] *= np.float32(2.0 ** -9)
    deq = w.astype(np.float32) * np.repeat(s, 64, axis=1)
    t = ((x - azp) * 0.02) @ deq.astype(np.float64).T
    q = (1 << ob) - 1
    so = float(np.abs(t).max()) / q * 1.5  # some outputs clip at either end
    ozp = q // 3
    want = np.clip(np.rint(t / so + ozp), 0, q)
    op = QuantMatmul(w, s, np.zeros(n, np.int32), act_bits=ab, out_bits=ob, act_scale=0.02, out_scale=so, act_zp=azp, out_zp=ozp,
                     weight_format=_lib.QH_WEIGHT_I4_GROUP, bias_float=np.zeros(n, np.float32), device=gpu)
    got = op(torch.from_numpy(x.astype(np.uint16 if ab == 16 else np.uint8)).to(gpu)).cpu().numpy()
    op.close()
    assert np.array_equal(got, want.astype(got.dtype)), f"{(got != want).sum()} of {got.size} differ"


@pytest.mark.parametrize("tie", [False, True], ids=["random", "ties"])
@pytest.mark.parametrize("mkn", REQUANT_SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("fam", C.GATED_FAMILIES)
def test_requantised_few_tiles(gpu, fam, mkn, tie):
    """Per-channel and LPBQ weights on the automatic path; with ties, power-of-two scales put odd
    dot products of the first rows exactly on half-integers (the float64 recomputation)."""
    import torch

    from qcom_htp_amd.qmm import QuantMatmul

    m, k, n = mkn
    c = C.synthetic_case(fam, m, k, n, seed=m + k, lpbq_block=32)
    if tie:
        rng = np.random.default_rng(n)
        zp, x = c.family.act_zp, c.activation_q.copy()
        for r in range(min(m, 40)):
            x[r] = zp
            pos = rng.choice(k, size=5, replace=False)
            x[r, pos] = zp + rng.integers(-3, 4, size=5)
        sA, s = 2.0 ** -7, 2.0 ** -8
        c = dataclasses.replace(c, activation_q=x, act_scale=sA, weight_scale=np.full(n, s, np.float32), out_scale=2.0 * sA * s,
                                weight_deq=c.weight_int_nk.astype(np.float32) * np.float32(s),
                                bias_q=rng.integers(-8, 8, size=n).astype(np.int32))
    op = QuantMatmul.from_case(c, device=gpu)
    got = op(torch.from_numpy(c.activation_q).to(gpu), out=unaligned(gpu, m, n, op.out_dtype)).cpu().numpy()
    op.close()
    want = oq.expected_output_case(c)
    assert np.array_equal(got, want), f"{(got != want).sum()} of {got.size} differ"


def test_more_tiles_than_one_launch_holds(gpu):
    """2^35 outputs: their 32 x 128 tiles of 512 threads are more than the 2^32 threads of a launch, so the
    rows are shared out over two.  The activations repeat every 64 rows, and so must the outputs."""
    import torch

    from qcom_htp_amd import _lib
    from qcom_htp_amd.qmm import QuantMatmul

    m, k, n, per = 65535 * 64, 32, 8224, 64
    if torch.cuda.mem_get_info(gpu)[0] < 2 * m * n * 3 // 2:
        pytest.skip("needs 104 GB of device memory")
    rng = np.random.default_rng(1)
    w = rng.integers(-32768, 32768, size=(n, k)).astype(np.int16)
    x = rng.integers(0, 65536, size=(per, k)).astype(np.uint16)
    op = QuantMatmul(w, np.ones(n, np.float32), np.zeros(n, np.int32), act_bits=16, out_bits=16, act_scale=1.0, out_scale=1.0,
                     act_zp=32768, out_zp=32768, weight_format=_lib.QH_WEIGHT_I16, device=gpu)
    act = torch.from_numpy(x.view(np.int16)).to(gpu).repeat(m // per, 1).view(torch.uint16)
    out = op.run_contract(act, "div_rint", 1 << 18).view(torch.int16).view(m // per, per * n)
    differ = sum(int((out[i:i + 4096] != out[0]).any(dim=1).sum()) for i in range(0, m // per, 4096))
    first = out[0].cpu().numpy().view(np.uint16).reshape(per, n)
    op.close()
    del out, act
    torch.cuda.empty_cache()
    assert np.array_equal(first, oq.contract_output(oq.int_accumulator(x, w, 32768), "div_rint", 1 << 18, None, 32768, 16))
    assert differ == 0, f"{differ} of {m // per} blocks of rows differ"
