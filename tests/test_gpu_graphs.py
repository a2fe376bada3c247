"""Compiled-graph parity on the MI355X: every benchmark configuration goes through
runtime::compile(graph, "hip") -> HipBackend::compile -> HipExecutable::run (the product path, C ABI kernels
underneath) and is compared with the same graph compiled for the oracle's `cpu` backend on identical seeded
inputs. Tolerances (stated per test) follow the north star: rtol 1e-5 for float32, 1e-2 for bfloat16, with
atol = rtol * rms(expected) (tests/tolerance.py). Full-size configurations that the single-threaded oracle
cannot finish in seconds are checked on sampled outputs recomputed with the oracle's per-element formula, or on
independent batch rows (each image / sequence of a batch is computed independently by every op on the path).
"""
import ctypes

import numpy as np
import pytest

import oracle_lib as orc
from frame_hip import graphs, host, synth
from tolerance import assert_bitwise, assert_close, assert_deep_lowp

pytestmark = pytest.mark.gpu
F32, F16, BF16 = 0, 2, 3


def say(msg):
    print(f"[case] {msg}", flush=True)


@pytest.fixture(scope="module")
def dev():
    n = host.device_count("hip")
    assert n >= 1, "no hip device"
    orc.load_cpu_backend()
    return n


def run_hip(g, ins, opt_level=1):
    return host.compile(g, "hip", opt_level).run(ins)


def retarget(g, device):
    return g.text().replace("@hip:0", f"@{device}:0")


# ---- HAL conformance (reference: tests/cpp/hal_conformance/test_hal_conformance.cpp:65-275) ---------------

def test_hal_conformance(dev):
    lib = host.lib()
    s = host.Stream("hip")
    ev = ctypes.c_void_p()
    host.check(lib.frame_event_create(b"hip", 0, ctypes.byref(ev)))
    host.check(lib.frame_event_synchronize(ev))  # never recorded: complete
    host.check(lib.frame_event_record(ev, s.handle))
    host.check(lib.frame_event_synchronize(ev))
    lib.frame_event_destroy(ev)
    a = np.arange(16, dtype=np.float32)  # 64 bytes through H2D / D2H
    t = host.Tensor.from_numpy("hip", F32, a)
    assert_bitwise(t.numpy(), a, "allocator round trip")
    assert t.data_ptr % 256 == 0


def test_eager_launch_add(dev):
    g = graphs.Graph("hip")
    x, y = g.input(F32, (1000,)), g.input(F32, (1000,))
    g.output(g.add(x, y))
    a, b = synth.tensor(1, (1000,), F32), synth.tensor(2, (1000,), F32)
    ta, tb = host.Tensor.from_numpy("hip", F32, a), host.Tensor.from_numpy("hip", F32, b)
    out = host.Tensor("hip", F32, (1000,))
    s = host.Stream("hip")
    host.launch(g.text(), "hip", [ta, tb], [out], s)
    s.synchronize()
    assert_bitwise(out.numpy(), a + b, "eager add")


# ---- C1 --------------------------------------------------------------------------------------------------

@pytest.mark.parametrize("batch", [64, 3])
def test_c1_mlp(dev, batch):
    say(f"C1 mlp f32 batch={batch}")
    g = graphs.mlp(batch=batch, dtype=F32, device="hip")
    ins = graphs.mlp_inputs(batch=batch, dtype=F32, seed=7)
    (got,) = run_hip(g, ins)
    (want,) = orc.run_graph_cpu(retarget(g, "cpu"), ins)
    assert_close(got, want, F32, what="C1 mlp")  # rtol 1e-5, atol 1e-5 * rms
    np.testing.assert_allclose(got.sum(1), 1.0, rtol=1e-5)


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_opt1_split_k_and_fusion_against_opt0(dev, dtype):
    # opt_level 1 folds add;relu / add into the GEMM epilogue and lets C1's small GEMMs sum k in four interleaved
    # quarters (the split-k kernel); opt_level 0 runs the unfused kernels in the reference's sequential order. The
    # two agree within the north star's rule, and each is within it of the oracle (softmax's exp differs from the
    # reference's in the last bits at either level).
    say(f"C1 opt1 vs opt0 dtype={dtype}")
    g = graphs.mlp(batch=64, dtype=dtype, device="hip")
    ins = graphs.mlp_inputs(batch=64, dtype=dtype, seed=9)
    lowered = host.hip_lowered(g.text(), 1)
    assert lowered.count("any_order=1") == 2, lowered
    o1, o0 = run_hip(g, ins, 1)[0], run_hip(g, ins, 0)[0]
    (want,) = orc.run_graph_cpu(retarget(g, "cpu"), ins)
    assert_close(o0, want, dtype, what="opt0 vs oracle")
    assert_close(o1, want, dtype, what="opt1 (split-k, fused) vs oracle")
    assert_close(o1, o0, dtype, what="opt1 vs opt0")


# ---- C2 --------------------------------------------------------------------------------------------------

@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("n", [1024, 2048, 4096])
def test_c2_gemm(dev, dtype, n):
    say(f"C2 gemm n={n} dtype={dtype}")
    g = graphs.gemm(n, dtype, device="hip")
    a, b = graphs.gemm_inputs(n, dtype)
    (got,) = run_hip(g, [a, b])
    if n == 1024:
        want = orc.matmul(dtype, a, b)
        assert_close(got, want, dtype, what=f"gemm {n}")
    else:
        rng = np.random.default_rng(n)
        rows, cols = rng.integers(0, n, 4096), rng.integers(0, n, 4096)
        want = orc.matmul_sample(dtype, a, b, rows, cols)
        # atol from the rms of the full product (U(-1,1) entries: rms = sqrt(n/9))
        assert_close(got[rows, cols], want, dtype, atol=(1e-5 if dtype == F32 else 1e-2) * np.sqrt(n / 9.0),
                     what=f"gemm {n} sampled")


def test_c2_gemm_odd_shapes(dev):
    for (m, k, n) in [(1, 1, 1), (7, 13, 5), (300, 264, 200), (17, 4096, 3), (65, 8, 1000)]:
        for dtype in (F32, BF16):
            say(f"gemm odd m={m} k={k} n={n} dtype={dtype}")
            g = graphs.gemm(n, dtype, device="hip", m=m, k=k)
            ins = graphs.gemm_inputs(n, dtype, m=m, k=k)
            assert_close(run_hip(g, ins)[0], orc.matmul(dtype, *ins), dtype, what=f"gemm {m}x{k}x{n}")


# ---- C3 --------------------------------------------------------------------------------------------------

@pytest.mark.parametrize("dtype", [F32, BF16])
def test_c3_conv_small_full(dev, dtype):
    for cfg in (dict(n=2, cin=64, h=12, w=12, cout=64, k=3), dict(n=2, cin=3, h=20, w=20, cout=16, k=7, stride=2, pad=3)):
        say(f"C3 conv small {cfg} dtype={dtype}")
        g = graphs.conv(dtype, device="hip", **cfg)
        ins = graphs.conv_inputs(dtype, n=cfg["n"], cin=cfg["cin"], h=cfg["h"], w=cfg["w"], cout=cfg["cout"], k=cfg["k"])
        (got,) = run_hip(g, ins)
        (want,) = orc.run_graph_cpu(retarget(g, "cpu"), ins)
        assert_close(got, want, dtype, what="conv small")


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_c3_conv_full_sampled(dev, dtype):
    say(f"C3 conv full dtype={dtype}")
    g = graphs.conv(dtype, device="hip")
    x, w, b = graphs.conv_inputs(dtype)
    (got,) = run_hip(g, [x, w, b])
    assert got.shape == (32, 64, 56, 56)
    idx = np.random.default_rng(3).integers(0, got.size, 4096)
    pre = orc.conv2d_sample(dtype, x, w, b, (32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1, 1), idx)
    want = orc.ew_program(dtype, [3], [1], [pre])  # relu after the rounded conv output
    assert_close(got.reshape(-1)[idx], want, dtype, atol=(1e-5 if dtype == F32 else 1e-2) * 1.4, what="conv C3 sampled")


# ---- C4 --------------------------------------------------------------------------------------------------

def resnet_f32_reference(batch, image, ins):
    """The same ResNet-18 graph in float32 on the CPU oracle, on the bf16 inputs' values."""
    g32, _ = graphs.resnet18(batch=batch, dtype=F32, device="cpu", image=image)
    (ref,) = orc.run_graph_cpu(g32, [synth.to_float(a, BF16).astype(np.float32) for a in ins])
    return ref


def test_c4_resnet_small_full(dev):
    # 20 bf16 conv layers: the tolerance is the deep-graph criterion of tests/tolerance.py (error vs a float32
    # evaluation: mean at most 1.25 x, max at most 2 x the bf16 oracle's own)
    say("C4 resnet18 bf16 batch=2 image=64")
    g, specs = graphs.resnet18(batch=2, dtype=BF16, device="hip", image=64)
    ins = graphs.resnet18_inputs(specs, batch=2, dtype=BF16, image=64)
    (got,) = run_hip(g, ins)
    (want,) = orc.run_graph_cpu(retarget(g, "cpu"), ins)
    stats = assert_deep_lowp(got, want, resnet_f32_reference(2, 64, ins), BF16, what="resnet18 64px")
    say(f"resnet18 64px error vs float32: {stats}")


def test_c4_resnet_full_rows(dev):
    # Full configuration on the GPU; the oracle recomputes images 0 and 1 (a batch-2 graph with the same weights
    # and the first two rows of the [64,1000] classifier bias).
    say("C4 resnet18 bf16 batch=64 image=224 (rows 0-1 checked)")
    g, specs = graphs.resnet18(batch=64, dtype=BF16, device="hip")
    ins = graphs.resnet18_inputs(specs, batch=64, dtype=BF16)
    (got,) = run_hip(g, ins)
    assert got.shape == (64, 1000) and np.isfinite(synth.to_float(got, BF16)).all()
    g2, specs2 = graphs.resnet18(batch=2, dtype=BF16, device="cpu")
    ins2 = [ins[0][:2]] + ins[1:-1] + [ins[-1][:2]]
    (want,) = orc.run_graph_cpu(g2, ins2)
    stats = assert_deep_lowp(got[:2], want, resnet_f32_reference(2, 224, ins2), BF16, what="resnet18 224px rows 0-1")
    say(f"resnet18 224px rows 0-1 error vs float32: {stats}")


# ---- C5 --------------------------------------------------------------------------------------------------

def test_c5_transformer_small_full(dev):
    say("C5 transformer bf16 small")
    g, shapes = graphs.transformer_block(batch=2, seq=64, d_model=128, heads=4, ffn=512, dtype=BF16, device="hip")
    ins = graphs.transformer_inputs(shapes, rows=128, d_model=128, dtype=BF16)
    (got,) = run_hip(g, ins)
    (want,) = orc.run_graph_cpu(retarget(g, "cpu"), ins)
    assert_close(got, want, BF16, what="transformer small")


@pytest.mark.parametrize("opt_level", [0, 1])
def test_c5_transformer_fused_attention(dev, opt_level):
    # head dim 64, so HipBackend::compile replaces the per-(batch, head) decomposition with one attention kernel
    say(f"C5 transformer bf16 batch=2 seq=128 heads=2 (fused attention) opt={opt_level}")
    g, shapes = graphs.transformer_block(batch=2, seq=128, d_model=128, heads=2, ffn=256, dtype=BF16, device="hip")
    lowered = host.hip_lowered(g.text(), opt_level)
    assert "hip_attention_internal" in lowered and "softmax" not in lowered
    # opt_level 1: the Q/K/V projections run as one grouped GEMM
    assert ("hip_matmul_grouped_internal" in lowered) == (opt_level == 1)
    ins = graphs.transformer_inputs(shapes, rows=256, d_model=128, dtype=BF16)
    (got,) = run_hip(g, ins, opt_level)
    (want,) = orc.run_graph_cpu(retarget(g, "cpu"), ins)
    assert_close(got, want, BF16, what="transformer with fused attention")


def test_c5_transformer_full_rows(dev):
    say("C5 transformer bf16 batch=8 seq=512 (sequences 0 and 7 checked)")
    g, shapes = graphs.transformer_block(dtype=BF16, device="hip")
    ins = graphs.transformer_inputs(shapes, dtype=BF16)
    (got,) = run_hip(g, ins)
    assert got.shape == (4096, 1024) and np.isfinite(synth.to_float(got, BF16)).all()
    g1, shapes1 = graphs.transformer_block(batch=1, dtype=BF16, device="cpu")
    # x and the full-shape biases (bq, bk, bv, bo, b1, b2) are per-row; weights and LayerNorm parameters are shared.
    # The first and the last sequence: the attention's and the biases' batch offsets are exercised at both ends.
    per_row = {0, 4, 6, 8, 10, 14, 16}
    for sq in (0, 7):
        rows = slice(512 * sq, 512 * (sq + 1))
        ins1 = [a[rows] if i in per_row else a for i, a in enumerate(ins)]
        (want,) = orc.run_graph_cpu(g1, ins1)
        assert_close(got[rows], want, BF16, what=f"transformer sequence {sq}")


# ---- graph replay (HipExecutable captures its steps on the second run with the same addresses) -----------------

@pytest.mark.parametrize("which", ["c1", "c5_small", "cnn_train"])
def test_graph_replay_matches_eager(dev, which, monkeypatch):
    """With FRAME_HIP_GRAPHS=1, run 1 is eager, run 2 captures a HIP graph and launches it, runs 3+ replay it. Between replays: new input
    values uploaded into the same tensors, another executable's eager work on the same stream, host syncs. Every
    replay must equal a fresh eager run of the same inputs bit for bit."""
    say(f"graph replay {which}")
    monkeypatch.setenv("FRAME_HIP_GRAPHS", "1")  # replay is opt-in; restored however the test ends
    if which == "c1":
        text = graphs.mlp(batch=64, dtype=F32, device="hip").text()
        make = lambda seed: graphs.mlp_inputs(batch=64, dtype=F32, seed=seed)
    elif which == "c5_small":
        g, shapes = graphs.transformer_block(batch=2, seq=128, d_model=256, heads=4, ffn=512, dtype=BF16)
        text = g.text()
        make = lambda seed: graphs.transformer_inputs(shapes, rows=256, d_model=256, dtype=BF16, seed=seed)
    else:
        g = graphs.cnn_train(batch=4, dtype=BF16)
        text = host.backward(g.text(), 0, [1, 2, 3, 4, 5, 6])
        make = lambda seed: graphs.cnn_train_inputs(batch=4, dtype=BF16, seed=seed)
    exe = host.compile(text, "hip")
    other = host.compile(graphs.gemm(256, BF16, device="hip").text(), "hip")
    other_ins = other.upload_inputs(graphs.gemm_inputs(256, BF16))
    other_outs = other.alloc_outputs()
    stream = host.Stream("hip")
    ins = exe.upload_inputs(make(11))
    outs = exe.alloc_outputs()
    for run in range(6):
        values = make(11 + run)
        for t, a in zip(ins, values):
            host.check(host.lib().frame_tensor_upload(t.handle, np.ascontiguousarray(a).ctypes.data, a.nbytes))
        exe.run_tensors(ins, outs, stream)  # eager, capture + launch, then replays
        other.run_tensors(other_ins, other_outs, stream)  # unrelated eager work on the same stream
        stream.synchronize()
        got = [o.numpy() for o in outs]
        want = host.compile(text, "hip").run(values)  # a fresh executable: eager
        for i, (a, b) in enumerate(zip(got, want)):
            assert_bitwise(a, b, f"{which} run {run} output {i}")
        if run in (2, 5):  # replays, checked against the oracle as well
            for i, (a, e) in enumerate(zip(got, orc.run_graph_cpu(text.replace("@hip:0", "@cpu:0"), values))):
                assert_close(np.asarray(a).reshape(-1), np.asarray(e).reshape(-1), F32 if which == "c1" else BF16,
                             what=f"{which} replay {run} output {i} vs oracle")


@pytest.mark.parametrize("elems", [1, 3])
def test_unaligned_caller_tensors(dev, elems):
    """Caller tensors that are views at an odd offset (Tensor::from_storage_slice): HipExecutable copies such inputs
    to aligned blocks and produces such outputs in blocks of its own, so C3 (the band conv, whose graph-layout filter
    path needs 16-byte aligned operands) and C1 give the same bits as with aligned tensors."""
    for name, g, ins in (("c3", graphs.conv(BF16, device="hip", n=2, cin=64, h=16, w=16, cout=64, k=3),
                          graphs.conv_inputs(BF16, n=2, cin=64, h=16, w=16, cout=64, k=3)),
                         ("c1", graphs.mlp(batch=64, dtype=F32, device="hip"), graphs.mlp_inputs(batch=64, dtype=F32))):
        say(f"unaligned caller tensors {name}, {elems} element(s) into their blocks")
        exe = host.compile(g, "hip")
        want = exe.run(ins)
        size = {F32: 4, F16: 2, BF16: 2}
        dt = [sp[0] for sp in exe.input_specs()]
        t_in = [host.Tensor.from_numpy("hip", d, a, byte_offset=elems * size[d]) for d, a in zip(dt, ins)]
        t_out = [host.Tensor("hip", d, shape, byte_offset=elems * size[d]) for d, shape in exe.output_specs()]
        assert all(t.data_ptr % 16 != 0 for t in t_in + t_out)
        stream = host.Stream("hip")
        for _ in range(2):
            exe.run_tensors(t_in, t_out, stream)
            stream.synchronize()
            for i, (o, w) in enumerate(zip(t_out, want)):
                assert_bitwise(o.numpy(), w, f"{name} unaligned output {i}")
