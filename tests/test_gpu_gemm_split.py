"""The tile GEMMs' bf16-split products at the sizes, alignments and values
where they can go wrong: partial tiles and stages, rows of fewer than four
elements, element-aligned operands (the general load form), int8 weights, and
values the split cannot hold (recomputed in fp32).

Tolerance: the operands are held exactly. Within a chunk of 64 the accumulator
takes at most 24 rounded terms per 16 k, then one per chunk is added to the
second; each rounding is at most 2^-23 of a partial sum (the matrix core
truncates) and independent, a standard deviation of 2^-23 / sqrt(12), so the
relative 2-norm error of a random product of many outputs stays below
sqrt(24 * 4 + K / 64) * 2^-24.8 (3.4e-7 at K = 64, 4.3e-7 at K = 4096; measured
1.1e-7 and 1.9e-7). A missing part product leaves 2e-6 and more, one accumulator
for a whole K = 4096 9e-7. A few outputs can all be small beside their terms, so
below 1000 of them the error is held against the terms."""
import ctypes as C
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

f32 = np.float32
LAYOUTS = ("gemm_nn", "gemm_nt", "gemm_tn")


@pytest.fixture(scope="module")
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from seeml_amd import _lib
    return torch, _lib.lib()


def device(torch, a, shift):
    """`a` on the GPU, `shift` elements past a 16-byte boundary."""
    buf = torch.zeros(a.size + 8, dtype=torch.from_numpy(a[:1]).dtype, device="cuda:0")
    view = buf[shift:shift + a.size]
    view.copy_(torch.from_numpy(a))
    return view


def call(gpu, name, *args):
    torch, L = gpu
    rc = getattr(L, "seeml_hip_" + name)(
        *[a.data_ptr() if hasattr(a, "data_ptr") else a for a in args],
        torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert rc == 0, L.seeml_hip_kernel_error().decode()


def bound(K):
    return np.sqrt(96 + K / 64) * 2.0 ** -24.8


def error_ok(got, A, B, scale=1.0, extra=0.0):
    """The bound on scale * A B, against the product or, for few outputs, its terms."""
    A, B = A.astype(np.float64), B.astype(np.float64)
    want = scale * (A @ B)
    size = want if want.size >= 1000 else scale * (np.abs(A) @ np.abs(B))
    return np.linalg.norm(got.reshape(want.shape) - want) <= (bound(A.shape[1]) + extra) * np.linalg.norm(size)


SIZES = [(1, 1, 1), (2, 3, 5), (3, 2, 64), (5, 130, 3), (130, 3, 17), (63, 65, 15), (65, 63, 33),
         (129, 131, 127), (257, 129, 66), (255, 259, 1027), (1000, 1531, 770)]


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("M,N,K", SIZES + [(192, 256, 4096)])
def test_any_extent_and_alignment(gpu, M, N, K, shift):
    """Every layout by the entry's own plan, and on both tiles of the general
    form (configs 0 and 5; the 16-byte form's where the size admits it)."""
    torch, _ = gpu
    r = np.random.default_rng([M, N, K])
    A, B = r.standard_normal((M, K), dtype=f32), r.standard_normal((K, N), dtype=f32)
    for layout, name in enumerate(LAYOUTS):
        a = device(torch, np.ascontiguousarray(A.T if layout == 2 else A).ravel(), shift)
        b = device(torch, np.ascontiguousarray(B.T if layout == 1 else B).ravel(), shift)
        for cfg in (None, 0, 5):
            out = torch.full((M * N + 4,), 7.0, device="cuda:0")
            if cfg is None:
                call(gpu, name, a, b, out[:M * N], M, N, K, *((None, 0) if layout == 0 else ()))
            else:
                call(gpu, "gemm_forced", layout, a, b, out[:M * N], M, N, K, cfg, 1)
            got = out.cpu().numpy()
            assert np.all(got[M * N:] == 7.0)
            assert error_ok(got[:M * N], A, B), (name, cfg)


@pytest.mark.parametrize("M,N,K", [(3, 5, 7), (65, 67, 33), (130, 258, 1030), (2048, 2048, 256),
                                   (2049, 1795, 643)])
def test_int8_weights(gpu, M, N, K):
    """The last two run the general form's 128x128 tile, the last at remainders."""
    torch, _ = gpu
    r = np.random.default_rng([M, N, K, 8])
    A = r.standard_normal((M, K), dtype=f32)
    B = r.integers(-128, 128, (K, N)).astype(np.int8)
    a, scale = device(torch, A.ravel(), 0), float(f32(0.01))
    for name, b in (("gemm_nn_q8", B), ("gemm_nt_q8", np.ascontiguousarray(B.T))):
        out = torch.empty(M * N, device="cuda:0")
        call(gpu, name, a, device(torch, b.ravel(), 3), out, M, N, K, scale,
             *((0,) if name == "gemm_nn_q8" else ()))
        # one more rounding: the scale's product
        assert error_ok(out.cpu().numpy(), A, B, scale, 2.0 ** -24), name


def special(kind, A, B):
    """A with row 70 carrying the value, B (its row 33 small, so that only the
    special term counts there), and what row 70 of the product must be."""
    bad, B = A.copy(), B.copy()
    if kind == "tiny":  # results around 1e-36
        bad[70] *= f32(1e-36)
    else:
        # int8 weights reach 128: past 2^103 all the same, with a finite product
        bad[70, 33] = {"inf": np.inf, "nan": np.nan, "huge": 1e36 if B.dtype == np.int8 else 3.4e38}[kind]
        B[33] = np.where(B[33] == 0, 1, B[33]) if B.dtype == np.int8 else B[33] * f32(1e-3)
    with np.errstate(all="ignore"):
        want = bad[70].astype(np.float64) @ B.astype(np.float64)
    return bad, B, np.sign(B[33].astype(np.float64)) * np.inf if kind == "inf" else want


def check_special(kind, got, want, clean, what):
    if kind == "nan":
        assert np.all(np.isnan(got[70])), what
    elif kind == "inf":
        assert np.array_equal(got[70], want), what
    else:
        assert np.linalg.norm(got[70] - want) <= 1e-6 * np.linalg.norm(want), what
    # rows outside the recomputed blocks (64..95) keep their bits
    keep = np.r_[0:64, 96:len(got)]
    assert np.array_equal(got[keep].view(np.uint32), clean[keep].view(np.uint32)), what


@pytest.mark.parametrize("kind", ["inf", "nan", "huge", "tiny"])
def test_values_the_split_cannot_hold(gpu, kind):
    """One row carries them; its block is recomputed in fp32 and every other
    output keeps its bits: every layout, tile config and split-K, the general
    form's tiles, int8 weights, scaled loads, groups and the LoRA epilogue.
    (The tiny row is within the split's range and must come out as well.)"""
    torch, L = gpu
    r = np.random.default_rng(9)
    host = lambda t, n: t.cpu().numpy().reshape(-1, n)  # noqa: E731
    empty = lambda n: torch.empty(n, device="cuda:0")  # noqa: E731
    for M, N, K, shift, cfgs in ((200, 136, 200, 0, range(L.seeml_hip_gemm_config_count() - 1)),
                                 (201, 137, 203, 1, (0, 5))):
        A, B = r.standard_normal((M, K), dtype=f32), r.standard_normal((K, N), dtype=f32)
        bad, B, want = special(kind, A, B)
        for layout in range(3):
            a, x = (device(torch, np.ascontiguousarray(v.T if layout == 2 else v).ravel(), shift) for v in (A, bad))
            b = device(torch, np.ascontiguousarray(B.T if layout == 1 else B).ravel(), shift)
            for splits in (1, 3):
                clean, first = empty(M * N), None
                call(gpu, "gemm_forced", layout, a, b, clean, M, N, K, 0, splits)
                for cfg in cfgs:
                    out = empty(M * N)
                    call(gpu, "gemm_forced", layout, x, b, out, M, N, K, cfg, splits)
                    got = host(out, N)
                    check_special(kind, got, want, host(clean, N), (layout, splits, cfg))
                    first = got if first is None else first
                    assert kind == "nan" or np.array_equal(got.view(np.uint32), first.view(np.uint32)), cfg
    # int8 weights
    M, N, K = 201, 137, 203
    A, Q = r.standard_normal((M, K), dtype=f32), r.integers(-128, 128, (K, N)).astype(np.int8)
    bad, Q, want = special(kind, A, Q)
    for name, q in (("gemm_nn_q8", Q), ("gemm_nt_q8", np.ascontiguousarray(Q.T))):
        outs = []
        for x in (A, bad):
            outs.append(empty(M * N))
            call(gpu, name, device(torch, x.ravel(), 0), device(torch, q.ravel(), 0), outs[-1], M, N, K,
                 2.0 ** -8, *((0,) if name == "gemm_nn_q8" else ()))
        check_special(kind, host(outs[1], N), want * 2.0 ** -8, host(outs[0], N), name)
    # scaled loads (NT, a rowdot shape), a group of two and the LoRA epilogue (NT)
    M, N, K, rank = 200, 64, 256, 16
    A, B = r.standard_normal((M, K), dtype=f32), r.standard_normal((K, N), dtype=f32)
    bad, B, want = special(kind, A, B)
    a, x, b = (device(torch, np.ascontiguousarray(v).ravel(), 0) for v in (A, bad, B.T))
    for cfg in (4, 5, 8, 9, 10, 11):
        outs = [empty(M * N), empty(M * N)]
        for o, v in zip(outs, (a, x)):
            call(gpu, "gemm_forced_scaled", 1, v, b, o, M, N, K, cfg, 1, 0.5)
        check_special(kind, host(outs[1], N), want * 0.5, host(outs[0], N), ("scaled", cfg))
    for cfg in (0, 1, 2, 3, 4, 5, 8, 9):
        outs = [empty(M * N), empty(M * N)]
        ptrs = lambda *ts: (C.c_void_p * 2)(*[t.data_ptr() for t in ts])  # noqa: E731
        call(gpu, "gemm_group", 1, cfg, 2, ptrs(a, x), ptrs(b, b), ptrs(*outs), (C.c_uint64 * 6)(*(M, N, K) * 2),
             None, None)
        check_special(kind, host(outs[1], N), want, host(outs[0], N), ("group", cfg))
    T, Bl = r.standard_normal((M, rank), dtype=f32), r.standard_normal((rank, N), dtype=f32)
    badT, wantT = T.copy(), None
    if kind == "tiny":
        badT[70] *= f32(1e-36)
    else:
        badT[70, 3] = {"inf": np.inf, "nan": np.nan, "huge": 3.4e38}[kind]
        Bl[3] *= f32(1e-3)
    with np.errstate(all="ignore"):
        wantT = np.sign(Bl[3].astype(np.float64)) * np.inf if kind == "inf" else badT[70].astype(np.float64) @ Bl
    zero = device(torch, np.zeros(M * K, f32), 0)
    for cfg in (0, 2, 4, 5, 8, 9):
        outs = [empty(M * N), empty(M * N)]
        for o, t in zip(outs, (T, badT)):
            call(gpu, "gemm_forced_lora", 1, zero, b, o, M, N, K, cfg, 0, 0, device(torch, t.ravel(), 0),
                 device(torch, Bl.ravel(), 0), rank, 0, 1.0, 1)
        check_special(kind, host(outs[1], N), wantT, host(outs[0], N), ("lora", cfg))


# Exponents of A's and B's values: A under bf16's smallest parts (2^-133) and
# subnormal, lifted by B; both small, with subnormal results; and operands and
# results past the scaled split's range (2^103, 2^80), which are recomputed.
RANGES = [(-112, 20), (-120, 24), (-126, 40), (-136, 60), (-146, 100), (30, -130), (-70, -70),
          (90, 20), (108, -30)]


def in_range(got, want, K, roundings=1):
    """The split's bound, or the fp32 MFMA's on recomputed blocks (K rounded
    terms), and `roundings` of fp32's smallest subnormal."""
    err = np.linalg.norm(got.astype(np.float64) - want)
    return err <= np.sqrt(96 + K) * 2.0 ** -24 * np.linalg.norm(want) + roundings * np.sqrt(want.size) * 2.0 ** -149


@pytest.mark.parametrize("ea,eb", RANGES)
def test_operands_of_every_magnitude(gpu, ea, eb):
    """Operands keep all 24 bits at every magnitude (subnormals those they
    have) whatever the other operand's, on every tile config, layout and load
    form, with split-K, int8 weights, scaled loads and in the LoRA epilogue."""
    torch, L = gpu
    r = np.random.default_rng([ea + 200, eb + 200])
    draw = lambda e, *shape: np.ldexp(r.standard_normal(shape), e).astype(f32)  # noqa: E731
    wide = lambda x: x.astype(np.float64)  # noqa: E731
    empty = lambda n: torch.full((n,), 7.0, device="cuda:0")  # noqa: E731
    M, N, K = 200, 136, 328
    A, B = draw(ea, M, K), draw(eb, K, N)
    want = wide(A) @ wide(B)
    for layout in range(3):
        a = device(torch, np.ascontiguousarray(A.T if layout == 2 else A).ravel(), 0)
        b = device(torch, np.ascontiguousarray(B.T if layout == 1 else B).ravel(), 0)
        for cfg in range(L.seeml_hip_gemm_config_count() - 1):
            for splits in (1, 3):
                out = empty(M * N)
                call(gpu, "gemm_forced", layout, a, b, out, M, N, K, cfg, splits)
                assert in_range(out.cpu().numpy().reshape(M, N), want, K, splits), (layout, cfg, splits)
    # the general form's two tiles
    for cfg in (0, 5):
        M, N, K = 131, 67, 77
        A, B = draw(ea, M, K), draw(eb, K, N)
        want = wide(A) @ wide(B)
        for layout in range(3):
            a = device(torch, np.ascontiguousarray(A.T if layout == 2 else A).ravel(), 1)
            b = device(torch, np.ascontiguousarray(B.T if layout == 1 else B).ravel(), 1)
            out = empty(M * N)
            call(gpu, "gemm_forced", layout, a, b, out, M, N, K, cfg, 1)
            assert in_range(out.cpu().numpy().reshape(M, N), want, K), (layout, cfg)
    # int8 weights under a scale of B's exponent
    Q, scale = r.integers(-128, 128, (K, N)).astype(np.int8), f32(np.ldexp(1.0, max(eb - 7, -120)))
    out = empty(M * N)
    call(gpu, "gemm_nn_q8", device(torch, A.ravel(), 0), device(torch, Q.ravel(), 0), out, M, N, K,
         float(scale), 0)
    assert in_range(out.cpu().numpy().reshape(M, N), float(scale) * (wide(A) @ wide(Q)), K, 1 + scale)
    # scaled loads: the factor brings the stream to A's exponent
    M, N, K, s = 256, 64, 328, f32(np.ldexp(0.75, max(ea, -140) // 2))
    A, B = draw(max(ea, -140) - max(ea, -140) // 2, M, K), draw(eb, N, K)
    for cfg in (4, 5, 8, 9, 10, 11):
        out = empty(M * N)
        call(gpu, "gemm_forced_scaled", 1, device(torch, A.ravel(), 0), device(torch, B.ravel(), 0), out,
             M, N, K, cfg, 1, float(s))
        assert in_range(out.cpu().numpy().reshape(M, N), wide(s * A) @ wide(B).T, K), cfg
    # the LoRA epilogue over a zero base product
    M, N, K, rank = 300, 264, 64, 16
    T, Bl = draw(ea, M, rank), draw(eb, rank, N)
    zero, w = device(torch, np.zeros(M * K, f32), 0), device(torch, draw(0, N, K).ravel(), 0)
    for cfg in (0, 2, 4, 5, 8, 9):
        out = empty(M * N)
        call(gpu, "gemm_forced_lora", 1, zero, w, out, M, N, K, cfg, 0, 0, device(torch, T.ravel(), 0),
             device(torch, Bl.ravel(), 0), rank, 0, 1.0, 1)
        assert in_range(out.cpu().numpy().reshape(M, N), wide(T) @ wide(Bl), rank), cfg


def test_narrow_outputs_take_narrow_tiles(gpu):
    """Every GEMM of this plan has an output at most 64 wide over 60000 rows:
    no tile may be wider than 64 both ways, however many of them there are."""
    from seeml_amd import DeviceUpdateEngine, PROGRAM_TRAIN, configs, planner
    cfg = planner.UpdateConfig(batch=60000, loss="xent", lr=1e-3,
                               lora=planner.LoraSpec(rank=8, alpha=16.0, seed=7))
    plan = planner.compile_update(configs.mlp_model(64, 64, 48), cfg)
    e = DeviceUpdateEngine(plan.blob)
    e.build()
    tiles = [re.search(r"(\d+)x(\d+)x\d+/", e.gemm_choice(PROGRAM_TRAIN, i)) for i in range(len(plan.train))]
    tiles = [(int(t[1]), int(t[2])) for t in tiles if t]
    assert tiles and all(min(t) <= 64 for t in tiles), tiles


@pytest.mark.parametrize("wide", [33, 48, 64])
def test_split_k_scratch_stays_within_the_covering_slices(gpu, wide):
    """A shape takes no more scratch than 128-deep slices covering the chip
    twice would: gemm_tn_noalloc serves every shape whose need by that count
    fits its array, with gemm_tn's bits."""
    from test_gpu_kernels import heuristic_splits
    torch, _ = gpu
    g = torch.Generator(device="cuda:0").manual_seed(wide)
    a, b = (torch.randn(8192 * 16400, device="cuda:0", generator=g) for _ in range(2))
    served = 0
    for other in (4097, 4801, 8193, 12290, 16399):
        for K in (1030, 4096, 8192):
            for M, N in ((wide, other), (other, wide)):
                if heuristic_splits(M, N, K) * M * N * 4 > 16 << 20:
                    continue
                want, got = (torch.empty(M * N, device="cuda:0") for _ in range(2))
                call(gpu, "gemm_tn", a, b, want, M, N, K)
                call(gpu, "gemm_tn_noalloc", a, b, got, M, N, K)
                assert torch.equal(got.view(torch.int32), want.view(torch.int32)), (M, N, K)
                served += 1
    assert served >= 6


@pytest.mark.parametrize("M,N,K", [(1024, 1024, 16), (1024, 1024, 64), (1024, 256, 4096)])
def test_errors_do_not_lean_to_one_side(gpu, M, N, K):
    """The mean error stays within ten standard deviations of the mean of that
    many independent errors, on every layout and tile config and in the LoRA
    epilogue: a lean would add up in a sum over rows."""
    torch, L = gpu
    g = torch.Generator(device="cuda:0").manual_seed(M + K)
    A, B = (torch.randn(*s, device="cuda:0", generator=g) for s in ((M, K), (K, N)))
    want = A.double() @ B.double()

    def check(out, what):
        e = out.reshape(M, N).double() - want
        assert float(e.mean().abs()) <= 10 * float(e.pow(2).mean().sqrt()) / (M * N) ** 0.5, what

    out = torch.empty(M * N, device="cuda:0")
    for layout in range(3):
        a, b = A.T.contiguous() if layout == 2 else A, B.T.contiguous() if layout == 1 else B
        for cfg in range(L.seeml_hip_gemm_config_count() - 1):
            call(gpu, "gemm_forced", layout, a, b, out, M, N, K, cfg, 1)
            check(out, (layout, cfg))
    if K == 16:
        zero, w = torch.zeros(M, 64, device="cuda:0"), torch.ones(N, 64, device="cuda:0")
        for cfg in (0, 2, 4, 5, 8, 9):
            call(gpu, "gemm_forced_lora", 1, zero, w, out, M, N, 64, cfg, 0, 0, A, B, K, 0, 1.0, 1)
            check(out, cfg)


def test_rows_four_million_elements_apart_keep_the_vector_form(gpu):
    """k-contiguous rows of 2^22 to 2^23 elements: 32-bit byte offsets reach 128
    of them, so a 256-row tile gives way to the 128-row one, in the 16-byte form
    that the LoRA epilogue needs."""
    torch, _ = gpu
    M, N, K, rank = 300, 64, (1 << 22) + 4, 16
    g = torch.Generator(device="cuda:0").manual_seed(5)
    A, B, T, Bl = (torch.randn(*s, device="cuda:0", generator=g) for s in ((M, K), (N, K), (M, rank), (rank, N)))
    out = torch.empty(M, N, device="cuda:0")
    call(gpu, "gemm_forced_lora", 1, A, B, out, M, N, K, 2, 0, 0, T, Bl, rank, 0, 1.0, 1)
    want = T.double() @ Bl.double()
    for k in range(0, K, 1 << 18):
        want += A[:, k:k + (1 << 18)].double() @ B[:, k:k + (1 << 18)].double().T
    # 2^16 chunk sums: bound(K), 1.5 times as the roundings of a growing sum are not alike
    assert float((out.double() - want).norm()) <= 1.5 * bound(K) * float(want.norm())
