"""GPU parity of the GDN chunk recurrence (stage B) and of the whole chunked prefill against the
float64 oracle (oracle.gdn.chunk_state_torch / gdn_prefill_torch, themselves pinned to the
token-by-token gated delta rule).

Error measure: relative Frobenius error per (batch, head) sequence, the oc of
scripts/gdn_solve_oc_check.py:31 applied to o [T, D] and to the final state S [D, D].
Bounds:
  stage B alone, W and U exact (float64 -> float32):
    QH_GDN_FP32  <= 1e-4   (hi/lo split products; the solve's fp32 bound)
    QH_GDN_BF16  <= 1.05e-2 (the bf16 bound of tests/qnn_kernel_e2e/correctness/test_gdn_solve_e2e.sh:18)
  prefill of few sequences (stage A + B): stage A is bf16-MFMA (qh_gdn_chunk_uw, bound 1.05e-2), so
  the whole path is held to 1.05e-2; of many (from T, no bf16 product in FP32): stage B's bounds.
"""

import numpy as np
import pytest

from oracle import gdn as og

pytestmark = pytest.mark.gpu

FP32_TOL = 1.0e-4
BF16_TOL = 1.05e-2


def bf16_bits(x):
    u = np.ascontiguousarray(x, dtype=np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def bits_f64(b):
    return (b.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def seq_inputs(B, T, H, seed):
    """q, k, v ~ N(0,1) as bf16 bits, beta = sigmoid(N(0,1)), gc = logsigmoid(N(0,1) + 3),
    [B, T, H, (D)] as the reference kernel takes them."""
    rng = np.random.default_rng(seed)
    qb, kb, vb = (bf16_bits(rng.standard_normal((B, T, H, 128))) for _ in range(3))
    beta = (1.0 / (1.0 + np.exp(-rng.standard_normal((B, T, H))))).astype(np.float32)
    gc = (-np.logaddexp(0.0, -(rng.standard_normal((B, T, H)) + 3.0))).astype(np.float32)
    return qb, kb, vb, beta, gc


def to_dev(x, gpu):
    import torch

    t = torch.from_numpy(np.ascontiguousarray(x))
    if x.dtype == np.uint16:
        t = t.view(torch.int16).view(torch.bfloat16)
    return t.to(gpu)


def per_seq(a):  # [B, T, H, D] -> [B*H, T, D]
    B, T, H, D = a.shape
    return np.ascontiguousarray(a.transpose(0, 2, 1, 3).reshape(B * H, T, D))


def worst_oc(x, ref, B, H):
    x = x.reshape(B * H, -1)
    ref = ref.reshape(B * H, -1)
    return max(og.oc(x[i], ref[i]) for i in range(B * H))


def stage_a_exact(kb, vb, beta, gc):
    """W (e^g form), U per 64-token chunk in float64 ([B, T, H, D])."""
    k64, v64 = bits_f64(kb), bits_f64(vb)
    B, T, H, D = k64.shape
    n = B * H * (T // 64)
    resh = lambda a: per_seq(a).reshape(n, 64, D)
    reshs = lambda a: np.ascontiguousarray(a.transpose(0, 2, 1).reshape(n, 64)).astype(np.float64)
    U, W = og.chunk_stage_a_torch(resh(k64), resh(v64), reshs(gc), reshs(beta), decay_w=True)
    back = lambda X: X.numpy().reshape(B, H, T, D).transpose(0, 2, 1, 3)
    return back(W), back(U)


@pytest.mark.parametrize("wu", ["f32", "bf16"], ids=["wu_f32", "wu_bf16"])
@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
@pytest.mark.parametrize("with_state", [False, True], ids=["zero_state", "incoming_state"])
@pytest.mark.parametrize("T", [192, 64], ids=["three_chunks", "one_chunk"])
def test_chunk_state_matches_fp64(gpu, precision, with_state, T, wu):
    """Stage B against the float64 recurrence; one chunk runs only the first (peeled) chunk, whose
    next-chunk prefetch reloads itself.  W and U go in as float32 or as bf16 (the instantiation
    gdn_prefill uses for BF16); the oracle gets the same rounded values."""
    import torch

    from qcom_htp_amd.gdn import gdn_chunk_state

    B, H = 2, 3
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=21 + with_state)
    W, U = stage_a_exact(kb, vb, beta, gc)
    if wu == "f32":
        Wd, Ud = W.astype(np.float32), U.astype(np.float32)
        W_in, U_in = Wd.astype(np.float64), Ud.astype(np.float64)
    else:
        Wd, Ud = bf16_bits(W), bf16_bits(U)
        W_in, U_in = bits_f64(Wd), bits_f64(Ud)
    S0 = (np.random.default_rng(5).standard_normal((B, H, 128, 128)) * 0.05).astype(np.float32) if with_state else None
    print(f"[gdn-state] stage B T={T} precision={precision} state={with_state} wu={wu}", flush=True)
    o, S = gdn_chunk_state(to_dev(qb, gpu), to_dev(kb, gpu), to_dev(gc, gpu), to_dev(Wd, gpu),
                           to_dev(Ud, gpu), None if S0 is None else to_dev(S0, gpu),
                           precision=precision, out_dtype=torch.float32)
    torch.cuda.synchronize()
    o_ref, S_ref = og.chunk_state_torch(per_seq(bits_f64(qb)), per_seq(bits_f64(kb)),
                                        np.ascontiguousarray(gc.transpose(0, 2, 1).reshape(B * H, T)),
                                        per_seq(W_in), per_seq(U_in),
                                        None if S0 is None else S0.reshape(B * H, 128, 128), 64)
    eo = worst_oc(per_seq(o.cpu().numpy().astype(np.float64)), o_ref.numpy(), B, H)
    es = worst_oc(S.cpu().numpy().astype(np.float64).reshape(B * H, 128, 128), S_ref.numpy(), B, H)
    tol = FP32_TOL if precision == 0 else BF16_TOL
    print(f"[gdn-state] precision={precision} state={with_state} wu={wu}: worst oc(o)={eo:.3e} oc(S)={es:.3e}",
          flush=True)
    assert eo <= tol and es <= tol


@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
@pytest.mark.parametrize("T", [256, 100], ids=["whole_chunks", "ragged"])
def test_prefill_matches_fp64(gpu, T, precision):
    """The whole prefill; BF16 runs stage A with bf16 W, U and stage B on its bf16-W/U kernel."""
    import torch

    from qcom_htp_amd.gdn import gdn_prefill

    B, H = 2, 3
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=31 + T)
    print(f"[gdn-state] prefill T={T} precision={precision}", flush=True)
    o, S = gdn_prefill(to_dev(qb, gpu), to_dev(kb, gpu), to_dev(vb, gpu), to_dev(gc, gpu), to_dev(beta, gpu),
                       precision=precision, out_dtype=torch.float32)
    torch.cuda.synchronize()
    gcs = np.ascontiguousarray(gc.transpose(0, 2, 1).reshape(B * H, T))
    bts = np.ascontiguousarray(beta.transpose(0, 2, 1).reshape(B * H, T))
    o_ref, S_ref = og.gdn_prefill_torch(per_seq(bits_f64(qb)), per_seq(bits_f64(kb)), per_seq(bits_f64(vb)), gcs,
                                        bts, 64)
    assert o.shape == (B, T, H, 128)
    eo = worst_oc(per_seq(o.cpu().numpy().astype(np.float64)), o_ref.numpy(), B, H)
    es = worst_oc(S.cpu().numpy().astype(np.float64).reshape(B * H, 128, 128), S_ref.numpy(), B, H)
    print(f"[gdn-state] prefill T={T}: worst oc(o)={eo:.3e} oc(S)={es:.3e}", flush=True)
    assert eo <= BF16_TOL and es <= BF16_TOL


def test_state_handoff_equals_one_pass(gpu):
    """Two calls, the second starting from the first's final state, give the one-pass result
    (same chunks, same arithmetic: equal to float32 rounding of the state hand-off)."""
    import torch

    from qcom_htp_amd.gdn import gdn_chunk_state, gdn_chunk_uw

    B, T, H = 1, 256, 4
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=41)
    q, k, v, g, bt = (to_dev(x, gpu) for x in (qb, kb, vb, gc, beta))
    w, u = gdn_chunk_uw(k, v, g, bt, 64, decay_w=True, out_dtype=torch.float32)
    o_all, S_all = gdn_chunk_state(q, k, g, w, u, out_dtype=torch.float32)
    h = T // 2
    cut = lambda x: (x[:, :h].contiguous(), x[:, h:].contiguous())
    (q1, q2), (k1, k2), (g1, g2), (w1, w2), (u1, u2) = (cut(x) for x in (q, k, g, w, u))
    o1, S1 = gdn_chunk_state(q1, k1, g1, w1, u1, out_dtype=torch.float32)
    o2, S2 = gdn_chunk_state(q2, k2, g2, w2, u2, S1, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.equal(o1, o_all[:, :h])
    assert torch.equal(o2, o_all[:, h:])
    assert torch.equal(S2, S_all)


@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
def test_chunk_state_bf16_output_is_rounded_fp32_output(gpu, precision):
    """The bfloat16 output path (4 rows x 4 columns of each lane quad exchanged so that every lane
    stores 4 adjacent outputs of one row) gives the float32 output rounded to nearest even, element
    for element: the two kernels differ only in how o is stored."""
    import torch

    from qcom_htp_amd.gdn import gdn_chunk_state, gdn_chunk_uw

    B, T, H = 2, 192, 3
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=43)
    q, k, v, g, bt = (to_dev(x, gpu) for x in (qb, kb, vb, gc, beta))
    w, u = gdn_chunk_uw(k, v, g, bt, 64, decay_w=True, out_dtype=torch.float32)
    print(f"[gdn-state] bf16 output, precision={precision}", flush=True)
    o32, S32 = gdn_chunk_state(q, k, g, w, u, precision=precision, out_dtype=torch.float32)
    o16, S16 = gdn_chunk_state(q, k, g, w, u, precision=precision, out_dtype=torch.bfloat16)
    torch.cuda.synchronize()
    assert o16.dtype == torch.bfloat16 and o16.shape == o32.shape
    assert torch.equal(o16, o32.to(torch.bfloat16))
    assert torch.equal(S16, S32)


def test_chunk_state_rejects_bad_arguments(gpu):
    import torch

    from qcom_htp_amd import _lib

    B, T, H = 1, 64, 1
    x = torch.zeros((B, T, H, 128), dtype=torch.bfloat16, device=gpu)
    g = torch.zeros((B, T, H), dtype=torch.float32, device=gpu)
    s = torch.zeros((B, H, 128, 128), dtype=torch.float32, device=gpu)
    o = torch.zeros_like(x)
    L = _lib.lib()
    args = lambda tok, chunk, hd, sin: (x.data_ptr(), x.data_ptr(), g.data_ptr(), x.data_ptr(), x.data_ptr(), sin,
                                        s.data_ptr(), o.data_ptr(), B, tok, H, hd, chunk, 0, 0, 0)
    assert L.qh_gdn_chunk_state(*args(T, 128, 128, 0)) == _lib.QH_STATUS_SHAPE_UNSUPPORTED
    assert L.qh_gdn_chunk_state(*args(T, 64, 64, 0)) == _lib.QH_STATUS_SHAPE_UNSUPPORTED
    assert L.qh_gdn_chunk_state(*args(100, 64, 128, 0)) == _lib.QH_STATUS_SHAPE_UNSUPPORTED
    assert L.qh_gdn_chunk_state(*args(T, 64, 128, s.data_ptr())) == _lib.QH_STATUS_INVALID_ARGUMENT  # alias


def test_prefill_of_few_sequences_has_no_workspace(gpu):
    """qh_gdn_prefill refuses the sequences that stages A and B serve better."""
    import torch

    from qcom_htp_amd import _lib

    L, x = _lib.lib(), torch.zeros(1 << 16, device=gpu)
    assert L.qh_gdn_prefill_workspace(1, 64, 64, 0) == 0 and L.qh_gdn_prefill_workspace(1, 64, 65, 0) > 0
    p = x.data_ptr()
    assert L.qh_gdn_prefill(p, p, p, p, p, 0, p, p, 1, 64, 1, 128, 0, 0, p, x.numel() * 4, 0) == _lib.QH_STATUS_SHAPE_UNSUPPORTED


def test_chunk_state_with_a_short_workspace_leaves_it_alone(gpu):
    """A workspace one byte short is not written, and the results are those of a sufficient one."""
    import torch

    from qcom_htp_amd import _lib
    from qcom_htp_amd.gdn import gdn_chunk_state, gdn_chunk_uw

    B, T, H = 1, 256, 3
    q, k, v, bt, g = (to_dev(x, gpu) for x in seq_inputs(B, T, H, seed=91))
    w, u = gdn_chunk_uw(k, v, g, bt, 64, decay_w=True, out_dtype=torch.float32)
    want, s_want = gdn_chunk_state(q, k, g, w, u, out_dtype=torch.float32)
    L = _lib.lib()
    need = L.qh_gdn_chunk_state_workspace(B, T, H, 0)
    assert need > 0
    for size in (need - 1, 0):
        ws = torch.full((need,), 0x5A, dtype=torch.uint8, device=gpu)
        o, s = torch.empty_like(want), torch.empty_like(s_want)
        st = L.qh_gdn_chunk_state_ws(q.data_ptr(), k.data_ptr(), g.data_ptr(), w.data_ptr(), u.data_ptr(), 0, s.data_ptr(),
                                     o.data_ptr(), B, T, H, 128, 64, _lib.QH_GDN_OUT_F32 | _lib.QH_GDN_WU_F32, 0, ws.data_ptr(),
                                     size, torch.cuda.current_stream().cuda_stream)
        assert st == _lib.QH_STATUS_OK
        assert torch.equal(o, want) and torch.equal(s, s_want) and bool((ws == 0x5A).all())


def test_prefill_full_config5_every_sequence(gpu):
    """Config 5 at full size (B=8, T=4096, H=32, D=128; 64 chunks per sequence): the GPU prefill
    against the float64 oracle on all 256 (batch, head) sequences, o and the final state, one
    batch of 32 sequences at a time on the host."""
    import torch

    from qcom_htp_amd.gdn import gdn_prefill

    B, T, H = 8, 4096, 32
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=55)
    print("[gdn-state] prefill config 5 B=8 T=4096 H=32", flush=True)
    o, S = gdn_prefill(to_dev(qb, gpu), to_dev(kb, gpu), to_dev(vb, gpu), to_dev(gc, gpu), to_dev(beta, gpu),
                       out_dtype=torch.float32)
    torch.cuda.synchronize()
    o = o.cpu().numpy()
    S = S.cpu().numpy()
    worst_o = worst_s = 0.0
    for b in range(B):
        sl = lambda a: a[b:b + 1]
        q1, k1, v1 = (per_seq(bits_f64(sl(x))) for x in (qb, kb, vb))
        o_ref, S_ref = og.gdn_prefill_torch(q1, k1, v1, np.ascontiguousarray(gc[b].T).astype(np.float64),
                                            np.ascontiguousarray(beta[b].T).astype(np.float64), 64)
        o_ref, S_ref = o_ref.numpy(), S_ref.numpy()
        ob = per_seq(o[b:b + 1].astype(np.float64))
        eo = max(og.oc(ob[h], o_ref[h]) for h in range(H))
        es = max(og.oc(S[b, h].astype(np.float64), S_ref[h]) for h in range(H))
        worst_o, worst_s = max(worst_o, eo), max(worst_s, es)
        print(f"[gdn-state] config 5 batch {b}: worst oc(o)={eo:.3e} oc(S)={es:.3e}", flush=True)
        assert eo <= BF16_TOL and es <= BF16_TOL, f"batch {b}"
    print(f"[gdn-state] config 5, all 256 sequences: worst oc(o)={worst_o:.3e} oc(S)={worst_s:.3e}", flush=True)


def test_torch_ops_prefill_matches_direct(gpu):
    import torch

    from qcom_htp_amd import torch_ops  # noqa: F401 (registers torch.ops.qhtp)
    from qcom_htp_amd.gdn import gdn_prefill

    B, T, H = 1, 128, 2
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=61)
    args = [to_dev(x, gpu) for x in (qb, kb, vb, gc, beta)]
    o_op, S_op = torch.ops.qhtp.gdn_prefill(*args, None, 0, True)
    o_d, S_d = gdn_prefill(*args, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert torch.equal(o_op, o_d) and torch.equal(S_op, S_d)


def test_python_surface_rejects_host_or_foreign_tensors(gpu):
    """A host initial_state (its address would be dereferenced on the device) and inputs on another
    device are refused before any launch."""
    import torch

    from qcom_htp_amd.gdn import gdn_chunk_state, gdn_prefill

    B, T, H = 1, 64, 1
    x = torch.zeros((B, T, H, 128), dtype=torch.bfloat16, device=gpu)
    g = torch.zeros((B, T, H), dtype=torch.float32, device=gpu)
    s_host = torch.zeros((B, H, 128, 128), dtype=torch.float32)
    with pytest.raises(TypeError, match="initial_state"):
        gdn_chunk_state(x, x, g, x, x, s_host)
    with pytest.raises(TypeError, match="initial_state"):
        gdn_prefill(x, x, x, g, g, s_host)
    with pytest.raises(TypeError):
        gdn_chunk_state(x, x, g, x, x, [0.0])


def test_prefill_on_a_side_stream_matches_current_stream(gpu):
    """gdn_prefill with a side stream (its temporaries allocated on that stream) gives the
    current-stream result."""
    import torch

    from qcom_htp_amd.gdn import gdn_prefill

    B, T, H = 1, 100, 2
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=77)
    q, k, v, g, bt = (to_dev(x, gpu) for x in (qb, kb, vb, gc, beta))
    o0, s0 = gdn_prefill(q, k, v, g, bt)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    o1, s1 = gdn_prefill(q, k, v, g, bt, stream=side)
    torch.cuda.current_stream().wait_stream(side)
    _ = torch.empty((1 << 20,), device=gpu).fill_(1.0)  # reuse pressure on the current stream
    torch.cuda.synchronize()
    assert torch.equal(o0, o1) and torch.equal(s0, s1)


@pytest.mark.parametrize("out", ["f32", "bf16"])
@pytest.mark.parametrize("wu", ["f32", "bf16"], ids=["wu_f32", "wu_bf16"])
@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
def test_few_sequences_equal_many(gpu, precision, wu, out):
    """The column-sliced kernels of few sequences (8, 4 and 2 workgroups per sequence) form every sum
    in the order of the one-workgroup kernel: the same sequences give the same bits alone, in groups
    and in a launch of all of them."""
    import torch

    from qcom_htp_amd.gdn import gdn_chunk_state, gdn_chunk_uw

    B, T, H = 1, 192, 160
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=77)
    q, k, v, bt, g = (to_dev(x, gpu) for x in (qb, kb, vb, beta, gc))
    s0 = torch.randn((B, H, 128, 128), generator=torch.Generator(device=gpu).manual_seed(3), device=gpu)
    w, u = gdn_chunk_uw(k, v, g, bt, 64, decay_w=True, out_dtype=torch.float32 if wu == "f32" else torch.bfloat16)
    run = lambda sl: gdn_chunk_state(*(x[:, :, sl].contiguous() for x in (q, k, g, w, u)), s0[:, sl].contiguous(), precision,
                                     torch.float32 if out == "f32" else torch.bfloat16)
    o_all, s_all = run(slice(0, H))
    for lo, n in ((0, 1), (1, 9), (10, 33), (43, 64), (90, 65)):
        o, s = run(slice(lo, lo + n))
        assert torch.equal(o, o_all[:, :, lo:lo + n]), f"{n} sequences: o differs"
        assert torch.equal(s, s_all[:, lo:lo + n]), f"{n} sequences: S differs"


@pytest.mark.parametrize("out", ["f32", "bf16"])
@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
@pytest.mark.parametrize("H", [3, 70], ids=["few_sequences", "many_sequences"])
@pytest.mark.parametrize("T", [1, 16, 63, 65, 100, 177])
def test_ragged_prefill_equals_zero_padded(gpu, T, H, precision, out):
    """A last partial chunk gives the bits of the same tokens padded with zeros to whole chunks."""
    import torch

    from qcom_htp_amd.gdn import gdn_prefill

    B = 2
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=T + H)
    q, k, v, bt, g = (to_dev(x, gpu) for x in (qb, kb, vb, beta, gc))
    s0 = torch.randn((B, H, 128, 128), generator=torch.Generator(device=gpu).manual_seed(3), device=gpu)
    odt = torch.float32 if out == "f32" else torch.bfloat16
    pad = -T % 64
    P = torch.nn.functional.pad
    qp, kp, vp = (P(x, (0, 0, 0, 0, 0, pad)) for x in (q, k, v))
    o_ref, s_ref = gdn_prefill(qp, kp, vp, P(g, (0, 0, 0, pad)), P(bt, (0, 0, 0, pad)), s0, precision, odt)
    o, s = gdn_prefill(q, k, v, g, bt, s0, precision, odt)
    assert torch.equal(o, o_ref[:, :T]) and torch.equal(s, s_ref)


@pytest.mark.parametrize("out", ["f32", "bf16"])
@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
@pytest.mark.parametrize("route", ["wu_f32", "wu_bf16", "from_t"])
def test_one_chunk_of_many_sequences(gpu, route, precision, out):
    """The kernels without a next chunk give the bits of the looping ones: the first chunk of two, and S
    handed over after it."""
    import torch

    from qcom_htp_amd.gdn import gdn_chunk_state, gdn_chunk_uw, gdn_prefill

    B, T, H = 1, 128, 70
    q, k, v, bt, g = (to_dev(x, gpu) for x in seq_inputs(B, T, H, seed=19))
    s0 = torch.randn((B, H, 128, 128), generator=torch.Generator(device=gpu).manual_seed(3), device=gpu)
    odt = torch.float32 if out == "f32" else torch.bfloat16
    if route == "from_t":
        args, run = (q, k, v, g, bt), lambda a, s: gdn_prefill(*a, s, precision, odt)
    else:
        w, u = gdn_chunk_uw(k, v, g, bt, 64, decay_w=True, out_dtype=torch.float32 if route == "wu_f32" else torch.bfloat16)
        args, run = (q, k, g, w, u), lambda a, s: gdn_chunk_state(*a, s, precision, odt)
    o, S = run(args, s0)
    o1, S1 = run([x[:, :64].contiguous() for x in args], s0)
    o2, S2 = run([x[:, 64:].contiguous() for x in args], S1)
    assert torch.equal(o1, o[:, :64]) and torch.equal(o2, o[:, 64:]) and torch.equal(S2, S)


def test_ragged_prefill_takes_strided_and_unaligned_inputs(gpu):
    import torch

    from qcom_htp_amd.gdn import gdn_prefill

    B, T, H = 1, 70, 2
    q, k, v, bt, g = (to_dev(x, gpu) for x in seq_inputs(B, T, H, seed=5))
    want = gdn_prefill(q, k, v, g, bt)
    odd = torch.empty(k.numel() + 1, dtype=k.dtype, device=gpu)[1:].view(k.shape)  # 2-byte aligned
    odd.copy_(k)
    strided = torch.stack((v, v), dim=-1)[..., 0]
    got = gdn_prefill(q, odd, strided, torch.stack((g, g), dim=-1)[..., 0], bt)
    assert all(torch.equal(x, y) for x, y in zip(got, want))


@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
@pytest.mark.parametrize("H", [2, 80], ids=["few_sequences", "many_sequences"])
@pytest.mark.parametrize("token", [16, 47, 100])
def test_state_infinity_stays_behind_its_tile(gpu, token, H, precision):
    """An infinite U at one token reaches no output of an earlier 16-token tile (P is lower triangular)."""
    import torch

    from qcom_htp_amd.gdn import gdn_chunk_state, gdn_chunk_uw

    q, k, v, bt, g = (to_dev(x, gpu) for x in seq_inputs(1, 128, H, seed=token))
    w, u = gdn_chunk_uw(k, v, g, bt, 64, decay_w=True, out_dtype=torch.float32)
    want, _ = gdn_chunk_state(q, k, g, w, u, None, precision)
    u[:, token] = float("inf")
    got, _ = gdn_chunk_state(q, k, g, w, u, None, precision)
    first = token // 16 * 16
    assert torch.equal(got[:, :first], want[:, :first])
    assert not torch.isfinite(got[:, token]).all()


@pytest.mark.parametrize("out", ["f32", "bf16"])
@pytest.mark.parametrize("wu", ["f32", "bf16"], ids=["wu_f32", "wu_bf16"])
@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
@pytest.mark.parametrize("T", [192, 193, 250, 320])
def test_operands_formed_ahead_equal_in_recurrence(gpu, T, precision, wu, out):
    """Few sequences' chunk operands formed in a workspace before the recurrence (one and two column tiles
    per workgroup, partial last chunks) give the bits of the one-workgroup kernel."""
    import torch

    from qcom_htp_amd import _lib
    from qcom_htp_amd.gdn import _chunk_state, _chunk_uw

    H = 130
    q, k, v, bt, g = (to_dev(x, gpu) for x in seq_inputs(1, T, H, seed=T))
    s0 = torch.randn((1, H, 128, 128), generator=torch.Generator(device=gpu).manual_seed(3), device=gpu)
    flags = _lib.QH_GDN_RAGGED if T % 64 else 0
    odt = torch.float32 if out == "f32" else torch.bfloat16
    w, u = _chunk_uw(k, v, g, bt, 64, True, torch.float32 if wu == "f32" else torch.bfloat16, None, 0, flags)
    run = lambda sl: _chunk_state(*(x[:, :, sl].contiguous() for x in (q, k, g, w, u)), s0[:, sl].contiguous(), precision, odt,
                                  None, flags)
    assert _lib.lib().qh_gdn_chunk_state_workspace(1, T, H, precision) == 0
    o_all, s_all = run(slice(0, H))
    for lo, n in ((0, 1), (1, 9), (10, 32), (50, 33), (60, 64)):
        assert _lib.lib().qh_gdn_chunk_state_workspace(1, T, n, precision) > 0
        o, s = run(slice(lo, lo + n))
        assert torch.equal(o, o_all[:, :, lo:lo + n]), f"{n} sequences: o differs"
        assert torch.equal(s, s_all[:, lo:lo + n]), f"{n} sequences: S differs"


@pytest.mark.parametrize("out", ["f32", "bf16"])
@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
@pytest.mark.parametrize("T", [1, 17, 64, 127, 193])
def test_prefill_from_t_matches_fp64(gpu, T, precision, out):
    """Many sequences take the recurrence from T = (I - A)^-1: o and S against the float64 recurrence.  In
    FP32 every product is split, so the bound is that of stage B alone (1e-4; a bf16 o adds its own
    rounding, at most 2^-9 of each value); in BF16 it is the bf16 bound."""
    import torch

    from qcom_htp_amd import _lib
    from qcom_htp_amd.gdn import gdn_prefill

    B, H = 2, 40
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=31 + T)
    q, k, v, bt, g = (to_dev(x, gpu) for x in (qb, kb, vb, beta, gc))
    s0 = 0.1 * torch.randn((B, H, 128, 128), generator=torch.Generator(device=gpu).manual_seed(3), device=gpu)
    assert _lib.lib().qh_gdn_prefill_workspace(B, T, H, precision) > 0
    o, S = gdn_prefill(q, k, v, g, bt, s0, precision, torch.float32 if out == "f32" else torch.bfloat16)
    x = lambda a: a.double().cpu().transpose(1, 2).contiguous()  # noqa: E731  [B, H, T, ...]
    qd, kd, vd, bd, gd, St = x(q), x(k), x(v), x(bt), x(g), s0.double().cpu().clone()
    qd = qd / torch.sqrt((qd * qd).sum(-1, keepdim=True) + 1e-6) / 128 ** 0.5
    kd = kd / torch.sqrt((kd * kd).sum(-1, keepdim=True) + 1e-6)
    want = torch.empty_like(vd)
    for t in range(T):  # token by token
        St = St * torch.exp(gd[:, :, t])[..., None, None]
        kt = kd[:, :, t]
        d = bd[:, :, t, None] * (vd[:, :, t] - (St * kt[..., None]).sum(-2))
        St = St + kt[..., None] * d[..., None, :]
        want[:, :, t] = (St * qd[:, :, t, :, None]).sum(-2)
    rel = lambda a, b: float((a - b).norm() / b.norm())  # noqa: E731
    tol = FP32_TOL if precision == 0 else BF16_TOL
    eo, es = rel(x(o), want), rel(S.double().cpu(), St)
    print(f"[gdn-state] prefill from T, T={T} precision={precision} out={out}: oc(o)={eo:.3e} oc(S)={es:.3e}", flush=True)
    assert eo <= tol + (2.0 ** -9 if out == "bf16" else 0.0) and es <= tol


@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
@pytest.mark.parametrize("T", [64, 100, 256])
def test_prefill_from_t_is_no_less_exact_than_from_w_and_u(gpu, T, precision):
    """The route of many sequences against the one of few (stages A and B, W and U at the precision that
    gdn_prefill gives them) on the same sequences: the distance from float64 is no larger, neither of
    the first chunk (where v_new is U, rounded once) nor of later ones, nor of S."""
    import torch

    from qcom_htp_amd import _lib
    from qcom_htp_amd.gdn import _chunk_state, _chunk_uw, gdn_prefill

    B, H = 2, 40
    qb, kb, vb, beta, gc = seq_inputs(B, T, H, seed=83 + T)
    q, k, v, bt, g = (to_dev(x, gpu) for x in (qb, kb, vb, beta, gc))
    assert _lib.lib().qh_gdn_prefill_workspace(B, T, H, precision) > 0
    flags = _lib.QH_GDN_RAGGED if T % 64 else 0
    w, u = _chunk_uw(k, v, g, bt, 64, True, torch.bfloat16 if precision else torch.float32, None, 0, flags)
    wu = _chunk_state(q, k, g, w, u, None, precision, torch.float32, None, flags)
    ft = gdn_prefill(q, k, v, g, bt, precision=precision, out_dtype=torch.float32)
    per_head = lambda a: np.ascontiguousarray(a.transpose(0, 2, 1).reshape(B * H, T)).astype(np.float64)  # noqa: E731
    o_ref, S_ref = og.gdn_prefill_torch(per_seq(bits_f64(qb)), per_seq(bits_f64(kb)), per_seq(bits_f64(vb)), per_head(gc),
                                        per_head(beta), 64)

    def errors(o, S):
        o = per_seq(o.cpu().numpy().astype(np.float64))
        parts = [(o[:, :64], o_ref.numpy()[:, :64]), (S.cpu().numpy().astype(np.float64).reshape(B * H, 128, 128), S_ref.numpy())]
        if T > 64:
            parts.append((o[:, 64:], o_ref.numpy()[:, 64:]))
        return [og.oc(x, y) for x, y in parts]

    e_wu, e_t = errors(*wu), errors(*ft)
    print(f"[gdn-state] T={T} precision={precision}: from W, U {e_wu}, from T {e_t}", flush=True)
    assert all(t <= w for t, w in zip(e_t, e_wu)), f"from T {e_t}, from W and U {e_wu}"


@pytest.mark.parametrize("precision", [0, 1], ids=["fp32", "bf16"])
@pytest.mark.parametrize("what", ["k", "v"])
@pytest.mark.parametrize("T,token", [(128, 16), (128, 47), (100, 99), (81, 80)])
def test_prefill_from_t_infinity_stays_behind_its_tile(gpu, T, token, what, precision):
    """An infinite key or value of one token reaches no output of an earlier 16-token tile and no other
    head; of a value, no other column.  At the end of a partial chunk, whose missing rows repeat the last
    token, the result is still that of zero tokens."""
    import torch

    from qcom_htp_amd.gdn import gdn_prefill

    B, H, h, col = 1, 80, 7, 5
    q, k, v, bt, g = (to_dev(x, gpu) for x in seq_inputs(B, T, H, seed=token))
    want, s_want = gdn_prefill(q, k, v, g, bt, None, precision)
    (k if what == "k" else v)[0, token, h, col] = float("inf")
    got, s_got = gdn_prefill(q, k, v, g, bt, None, precision)
    same = torch.ones((T, H, 128), dtype=torch.bool, device=gpu)
    same[token // 16 * 16:, h] = False
    if what == "v":
        same[:, :, :col] = same[:, :, col + 1:] = True
    assert torch.equal(got[0][same], want[0][same])
    assert not torch.isfinite(got[0, token, h, col])
    heads = torch.arange(H, device=gpu) != h
    assert torch.equal(s_got[:, heads], s_want[:, heads]) and not torch.isfinite(s_got[0, h, :, col]).any()
    P, pad = torch.nn.functional.pad, -T % 64
    qp, kp, vp = (P(x, (0, 0, 0, 0, 0, pad)) for x in (q, k, v))
    o_pad, s_pad = gdn_prefill(qp, kp, vp, P(g, (0, 0, 0, pad)), P(bt, (0, 0, 0, pad)), None, precision)
    for x, y in ((got, o_pad[:, :T]), (s_got, s_pad)):
        assert torch.equal(torch.isnan(x), torch.isnan(y)) and torch.equal(torch.nan_to_num(x), torch.nan_to_num(y))
