"""GPU parity of the GEMM families against the oracle (fp32 dequantize-then-matmul, f64 for the MQA logits).

fp8 GEMMs: every test prints a PARITY line with the stated bar's measures against bf16(fp32 reference):
rel-L2 (required <= 1e-3), the largest |out - bf16(ref)| in bf16 ulps, and the elements above 2 bf16 ulp plus
the f32 accumulation-order noise (k/64 + 32) 2^-24 sum|a w|.  The fp8 MFMA does not round its 64-product dot
exactly (it truncates each group of 8 products to 13 bits below the group's largest exponent, see
oracle/kg_oracle.c kgo_mfma_f8, pinned on the GPU by tests/test_gpu_mfma_kat.py), so a few elements can sit
above that bar; the same line therefore compares the output with the oracle's model of the instruction, as the
kernels sequence it (oracle.ref.fp8_gemm_mfma), which it must equal on >= 99.9% of the elements and match within
1 bf16 ulp everywhere.  bf16 GEMMs must meet the stated bar on every element.  MQA logits (f32) within
(128 + 32 + 16) 2^-24 sum_h |w| ksf sum_d |q k| plus 2^-7 times the instruction's window bound.
Every test also checks that memory the op must not write (columns past n, rows past m, rows no expert
owns, the rope columns next to W_UK's output, logits past a row's key count) is left untouched."""
import numpy as np
import pytest
import torch

from kern_glm53_amd import ops, synth
from oracle import ref
from tests._gpu import DEV, bf16_bits, d, fastest, filled, h

pytestmark = pytest.mark.gpu

SENTINEL = 0x7fc1            # a bf16 NaN pattern no kernel produces


def quant_act(M, K, rows, lda, sfa_rows, seed):
    """Activation operand: e4m3 [rows][lda] (rows >= M zero) and scale words [K/512][sfa_rows]."""
    x = bf16_bits(synth.activations(M, K, synth.generator(seed)))
    a = np.zeros((rows, lda), np.uint8)
    sfa = np.zeros(ref.sf_words(K) * sfa_rows * 4, np.uint8)
    q, _ = ref.quant(x, K, sfa_rows, M, None, sfa)
    a[:M, :K] = q
    return a, sfa


def quant_weight(N, K, seed, groups=1):
    """Weight operand through the requant math: e4m3 [groups*N][K], scale words [groups*K/512][N]."""
    w8, s = synth.weights(groups * N, K, synth.generator(seed))
    w8, s = w8.numpy(), s.numpy()
    wq = np.zeros((groups * N, K), np.uint8)
    kw = ref.sf_words(K)
    sfb = np.zeros(groups * kw * N * 4, np.uint8)
    gr = (N + 127) // 128 * 128 if groups == 1 else N
    ref.requant(w8, s, wq, sfb, groups * N, K, gr, N if groups > 1 else 0, 0, N, kw * N if groups > 1 else 0)
    return wq, sfb


def check(out_bits, ref32, abs_sum, k, what, model=None, window=None):
    """The parity bar (module docstring); prints the measured PARITY line."""
    out = torch.from_numpy(out_bits.view(np.int16)).view(torch.bfloat16).float()
    ok, rep = ref.check_bf16_gemm(out, ref32, abs_sum, k, model32=model, window=window)
    line = ref.parity_line(what, rep)
    print(line, flush=True)
    assert ok, line
    return rep


def sample_rows(M, extra=12, seed=0):
    """Rows the MFMA model is evaluated on for large GEMMs: tile edges and random rows."""
    if M <= 64:
        return np.arange(M)
    edge = {0, 1, 127, 128, 255, 256, M // 2, M - 2, M - 1}
    rnd = np.random.default_rng(seed).choice(M, extra, replace=False).tolist()
    return np.array(sorted(r for r in edge | set(rnd) if 0 <= r < M))


def model_on_rows(a, w, sfa, sfb, M, N, K, lda, sfa_rows, rows):
    """fp8_gemm_mfma on `rows` of a dense GEMM, NaN on the other rows."""
    out = np.full((M, N), np.nan, np.float32)
    a_s = np.ascontiguousarray(np.asarray(a).reshape(-1, lda)[rows])
    sfa_s = np.ascontiguousarray(np.asarray(sfa).reshape(-1, sfa_rows, 4)[:, rows, :])
    out[rows] = ref.fp8_gemm_mfma(a_s, w, sfa_s, sfb, len(rows), N, K, lda, len(rows))
    return out


# ------------------------------------------------------------------ dense (a2)

# the persistent 256 x 256 kernel with row tails of 1-128 (half tiles) and 129-255 rows, column tails, and more K blocks
# than one scale word holds (the picks are checked in test_dispatch.py)
PERSISTENT = [
    (4100, 3080, 1152, 4224, 1152, 3088, 4224),     # a row tail of 4, a column tail of 8, 9 K blocks
    (1900, 6152, 896, 1900, 912, 6160, 1910),       # a row tail of 108, 7 K blocks, lda > k
    (4000, 2632, 1536, 4096, 1536, 2632, 4096),     # a row tail of 160, 12 K blocks
    (2300, 4168, 640, 2304, 640, 4176, 2300 + 8),   # a row tail of 252, 5 K blocks
    (4000, 4160, 640, 4096, 640, 4224, 4096),
    (4352, 4224, 896, 4352, 896, 4232, 4352),       # 17 x 17 tiles, a column tail of 128
]


@pytest.mark.parametrize("M,N,K,rows,lda,ldc,sfa_rows", [
    (512, 2048, 6144, 512, 6144, 2048, 512),        # the parity configuration
    (300, 2624, 1024, 320, 1152, 2752, 384),        # N tail of 64 (2624 = 20.5 x 128), ldc > n, lda > k
    (4096, 4096, 512, 4096, 512, 4096, 4096),       # 256 x 256 tiles
    (4100, 4096, 1536, 4224, 1536, 4096, 4224),     # 128 x 192 tiles, an M tail of 4 rows, K = 3 x 512
    (4096, 4096, 128, 4096, 128, 4096, 4096),       # one K block: three padded stages of four
    (8192, 2048, 2560, 8192, 2560, 2048, 8192),     # K = 5 groups of four stages
    (512, 256, 384, 512, 384, 256, 512),            # odd K-block count, 32 x 32 tiles
    (1, 2048, 6144, 16, 6144, 2048, 16),            # a single row
] + PERSISTENT)
def test_fp8_gemm(M, N, K, rows, lda, ldc, sfa_rows):
    a, sfa = quant_act(M, K, rows, lda, sfa_rows, seed=M + N + K)
    w, sfb = quant_weight(N, K, seed=N * 7 + K)
    ref32 = ref.fp8_gemm(a, w, sfa, sfb, M, N, K, lda, sfa_rows)
    S = ref.fp8_gemm_abs(a, w, sfa, sfb, M, N, K, lda, sfa_rows)
    # the MFMA model on every row of the parity configuration, on sampled rows of the others
    rows_m = np.arange(M) if (M, N, K) == (512, 2048, 6144) else sample_rows(M, seed=M + N)
    model = model_on_rows(a, w, sfa, sfb, M, N, K, lda, sfa_rows, rows_m)
    c = filled((rows, ldc), SENTINEL, torch.int16)
    window = ref.fp8_window_bound(a, w, sfa, sfb, M, N, K, lda, sfa_rows)
    ops.fp8_gemm(d(a), d(w), d(sfa), d(sfb), c, M, n=N, k=K, rows=rows, lda=lda, ldc=ldc, sfa_rows=sfa_rows)
    out = h(c, np.uint16)
    check(np.ascontiguousarray(out[:M, :N]), ref32, S, K, f"dense {M}x{N}x{K}", model, window)
    assert np.all(out[:M, N:] == SENTINEL) and np.all(out[M:] == SENTINEL)


# (rows, columns, workgroups a CU) of the tile -> sizes that the dense GEMM runs in it, with C rows of an odd stride
TILE_SHAPES = {
    (32, 32, 1): [(1, 5, 128), (31, 100, 640), (33, 97, 2176)],     # one K block, odd block counts, past a ring
    (64, 64, 1): [(200, 1201, 384), (193, 1216, 1152)],
    (64, 128, 1): [(640, 1700, 128), (577, 1729, 1408)],
    (128, 128, 1): [(1000, 2500, 384), (897, 2433, 640)],
    (128, 192, 1): [(1500, 3300, 384), (1409, 3265, 1664)],         # fewer K blocks than stages, past a loop body
    (128, 128, 2): [(2000, 3700, 256)],
}


@pytest.mark.parametrize("M,N,K", [size for sizes in TILE_SHAPES.values() for size in sizes])
def test_fp8_gemm_tile_shapes(M, N, K):
    """Each tile shape the dense GEMM picks by size (test_dispatch.py checks the picks), with row, column and K
    remainders: sampled rows against the oracle and its MFMA model at the bar of test_fp8_gemm, nothing written past m and n."""
    print(f"fp8 gemm {M}x{N}x{K}", flush=True)
    ldc = (N + 3) // 4 * 4 + 4
    a, sfa = quant_act(M, K, M, K, M, seed=M + 5 * N + K)
    w, sfb = quant_weight(N, K, seed=N + 3 * K)
    c = filled((M + 2, ldc), SENTINEL, torch.int16)
    ops.fp8_gemm(d(a), d(w), d(sfa), d(sfb), c, M, n=N, k=K, rows=M, lda=K, ldc=ldc, sfa_rows=M)
    out = h(c, np.uint16)
    rs = sample_rows(M, seed=M)
    R = len(rs)
    a_s = np.ascontiguousarray(a[rs])
    sfa_s = np.ascontiguousarray(sfa.reshape(-1, M, 4)[:, rs, :]).reshape(-1)
    ref32 = ref.fp8_gemm(a_s, w, sfa_s, sfb, R, N, K, K, R)
    S = ref.fp8_gemm_abs(a_s, w, sfa_s, sfb, R, N, K, K, R)
    model = ref.fp8_gemm_mfma(a_s, w, sfa_s, sfb, R, N, K, K, R)
    window = ref.fp8_window_bound(a_s, w, sfa_s, sfb, R, N, K, K, R)
    check(np.ascontiguousarray(out[rs, :N]), ref32, S, K, f"dense {M}x{N}x{K}", model, window)
    assert np.all(out[:M, N:] == SENTINEL) and np.all(out[M:] == SENTINEL)


@pytest.mark.parametrize("M,N,K", [(4200, 4096, 1024), (5000, 2752, 6144), (2300, 6144, 16384), (11000, 1024, 512)])
def test_fp8_gemm_pick_time(M, N, K):
    """Dense GEMMs that 256 x 256 tiles cover in one round, or in two where the smaller tiles need three, are no slower
    than the grouped entry point's 256 x 256 tiles over the same rows as one expert (they took 1.25 to 1.5 times it), and
    equal it."""
    g = synth.generator(M + N, "cuda")
    rows = (M + 127) // 128 * 128
    codes = lambda *s: torch.randint(0, 0x78, s, generator=g, device=DEV, dtype=torch.uint8)
    sf = lambda r: torch.randint(118, 127, (ref.sf_words(K) * r * 4,), generator=g, device=DEV, dtype=torch.uint8)
    a, w, sfa, sfb = codes(rows, K), codes(N, K), sf(rows), sf(N)
    psum = torch.tensor([M], dtype=torch.int32, device=DEV)
    c0, c1 = filled((rows, N), SENTINEL, torch.int16), filled((rows, N), SENTINEL, torch.int16)
    dense, grouped = fastest([lambda: ops.fp8_gemm(a, w, sfa, sfb, c0, M, n=N, k=K, rows=rows, lda=K, ldc=N, sfa_rows=rows),
                              lambda: ops.fp8_gemm_psum(a, w, sfa, sfb, c1, psum, n=N, k=K, rows=rows, lda=K, ldc=N,
                                                        sfa_rows=rows, groups=1)])
    print(f"dense {M}x{N}x{K}: {dense:.1f} us, as one group {grouped:.1f}", flush=True)
    assert torch.equal(c0, c1)
    assert dense <= 1.15 * grouped


@pytest.mark.parametrize("N,K,ldc", [(2624, 6144, 2752), (16384, 2048, 20480), (6144, 16384, 6144)])
def test_fp8_gemm_bench_shapes_sampled(N, K, ldc):
    """The bench's dense GEMMs at full size (M = 16384: q_a/kv_a, q_b, o_proj): activations quantized on the
    GPU by glm_quant (bit-exact against the oracle elsewhere), random e4m3 weights and UE8M0 scales; 16
    output rows (tile edges and random ones) against the oracle's dequantize-then-matmul, every column."""
    M = 16384
    print(f"fp8 gemm 16384 x {N} x {K}", flush=True)
    g = synth.generator(N + K, "cuda")
    x = synth.activations(M, K, g, device="cuda")
    q = torch.empty(M, K, dtype=torch.uint8, device=DEV)
    sf = torch.empty(ref.sf_words(K) * M * 4, dtype=torch.uint8, device=DEV)
    ops.quant(x, K, q, sf, M, K, M)
    w = torch.randint(0, 256, (N, K), generator=g, device=DEV, dtype=torch.int32)
    w = torch.where((w & 0x7f) == 0x7f, w ^ 1, w).to(torch.uint8)            # no NaN codes
    sfb = torch.randint(118, 127, (ref.sf_words(K) * N * 4,), generator=g, device=DEV, dtype=torch.int32)
    sfb = sfb.to(torch.uint8)
    c = torch.full((M, ldc), -7.0, dtype=torch.bfloat16, device=DEV)
    ops.fp8_gemm(q, w, sf, sfb, c, M, n=N, k=K, rows=M, lda=K, ldc=ldc, sfa_rows=M)
    rows = sorted({0, 1, 255, 256, 8191, 8192, 16127, 16383} |
                  set(np.random.default_rng(N).choice(M, 8, replace=False).tolist()))
    R = len(rows)
    a_s = h(q[rows], np.uint8)
    sfa_s = np.ascontiguousarray(h(sf, np.uint8).reshape(-1, M, 4)[:, rows, :]).reshape(-1)
    w_h, sfb_h = h(w, np.uint8), h(sfb, np.uint8)
    ref32 = ref.fp8_gemm(a_s, w_h, sfa_s, sfb_h, R, N, K, K, R)
    S = ref.fp8_gemm_abs(a_s, w_h, sfa_s, sfb_h, R, N, K, K, R)
    model = ref.fp8_gemm_mfma(a_s, w_h, sfa_s, sfb_h, R, N, K, K, R)
    window = ref.fp8_window_bound(a_s, w_h, sfa_s, sfb_h, R, N, K, K, R)
    out = h(c.view(torch.int16), np.uint16)
    check(np.ascontiguousarray(out[rows, :N]), ref32, S, K, f"dense 16384x{N}x{K} ({R} rows)", model, window)
    assert np.all(out[rows, N:] == 0xc0e0)                                     # bf16 -7.0 past n untouched


def test_fp8_gemm_scale_linearity():
    """Raising one activation row's exponent bytes by 3 multiplies exactly that output row by 8 (the
    kernel applies the UE8M0 scales exactly)."""
    M, N, K = 256, 512, 1024
    a, sfa = quant_act(M, K, M, K, M, seed=21)
    w, sfb = quant_weight(N, K, seed=22)
    c1 = torch.empty(M, N, dtype=torch.int16, device=DEV)
    c2 = torch.empty(M, N, dtype=torch.int16, device=DEV)
    ops.fp8_gemm(d(a), d(w), d(sfa), d(sfb), c1, M, n=N, k=K, rows=M, lda=K, ldc=N, sfa_rows=M)
    sfa2 = sfa.copy()
    for kb in range(K // 128):
        sfa2[((kb >> 2) * M + 17) * 4 + (kb & 3)] += 3
    ops.fp8_gemm(d(a), d(w), d(sfa2), d(sfb), c2, M, n=N, k=K, rows=M, lda=K, ldc=N, sfa_rows=M)
    o1 = c1.view(torch.bfloat16).float().cpu()
    o2 = c2.view(torch.bfloat16).float().cpu()
    assert torch.equal(o2[17], o1[17] * 8)
    o1[17] = 0
    o2[17] = 0
    assert torch.equal(o1, o2)


# ------------------------------------------------------------------ m-grouped psum (a3)

EDGE = [0, 1, 127, 128, 129, 256, 255, 383, 2, 0, 64]


def grouped_case(T, n, k, seed):
    counts = list(EDGE) + [0] * (256 - len(EDGE))
    rest = T * 8 - sum(counts)
    for e in range(len(EDGE), 256):
        counts[e] = rest // (256 - len(EDGE))
    counts[255] += T * 8 - sum(counts)
    counts = np.array(counts, np.int32)
    psum = ref.moe_psum(counts)
    rows = 8 * T + 256 * 128
    a, sfa = quant_act(rows, k, rows, k, rows, seed=seed)
    w, sfb = quant_weight(n, k, seed=seed + 1, groups=256)
    return counts, psum, rows, a, sfa, w, sfb


@pytest.mark.parametrize("n,k", [(512, 512), (384, 640)])
def test_fp8_gemm_psum(n, k):
    T = 256
    counts, psum, rows, a, sfa, w, sfb = grouped_case(T, n, k, seed=n + k)
    ref32, S = ref.fp8_gemm_psum(a, w, sfa, sfb, psum, 256, n, k, rows, k, rows, abs_too=True)
    model = ref.fp8_gemm_psum_mfma(a, w, sfa, sfb, psum, 256, n, k, rows, k, rows)
    window = ref.fp8_gemm_psum_window(a, w, sfa, sfb, psum, 256, n, k, rows, k, rows)
    c = filled((rows, n), SENTINEL, torch.int16)
    ops.fp8_gemm_psum(d(a), d(w), d(sfa), d(sfb), c, d(psum), n=n, k=k, rows=rows, lda=k, ldc=n, sfa_rows=rows)
    out = h(c, np.uint16)
    owned = ~torch.isnan(ref32[:, 0]).numpy()
    check(np.ascontiguousarray(out[owned]), ref32[owned], S[owned], k, f"psum n={n} k={k}", model[owned],
          window[owned])
    assert np.all(out[~owned] == SENTINEL)


@pytest.mark.parametrize("groups,seed", [(8, 61), (1024, 62)])
def test_fp8_gemm_psum_groups(groups, seed):
    """Other expert counts: 8 large groups (many full row tiles per expert, several tiles per CU), and the
    maximum of 1024 with most groups empty and tails of every size."""
    n, k = 256, 512
    rng = np.random.default_rng(seed)
    if groups == 8:
        counts = np.array([2300, 0, 129, 4097, 511, 1, 768, 1500], np.int32)
    else:
        counts = np.where(rng.random(groups) < 0.3, rng.integers(1, 400, groups), 0).astype(np.int32)
    psum = ref.moe_psum(counts, groups)
    rows = int((psum[-1] + 127) // 128 * 128) + 256
    a, sfa = quant_act(rows, k, rows, k, rows, seed=seed)
    w, sfb = quant_weight(n, k, seed=seed + 1, groups=groups)
    ref32, S = ref.fp8_gemm_psum(a, w, sfa, sfb, psum, groups, n, k, rows, k, rows, abs_too=True)
    model = ref.fp8_gemm_psum_mfma(a, w, sfa, sfb, psum, groups, n, k, rows, k, rows)
    window = ref.fp8_gemm_psum_window(a, w, sfa, sfb, psum, groups, n, k, rows, k, rows)
    c = filled((rows, n), SENTINEL, torch.int16)
    ops.fp8_gemm_psum(d(a), d(w), d(sfa), d(sfb), c, d(psum), n=n, k=k, rows=rows, lda=k, ldc=n, sfa_rows=rows,
                      groups=groups)
    out = h(c, np.uint16)
    owned = ~torch.isnan(ref32[:, 0]).numpy()
    check(np.ascontiguousarray(out[owned]), ref32[owned], S[owned], k, f"psum groups={groups}", model[owned],
          window[owned])
    assert np.all(out[~owned] == SENTINEL)


@pytest.mark.parametrize("wide", [False, True])
def test_fp8_gemm_psum_silu_quant_matches_unfused_chain(wide):
    """The fused epilogue equals gate_up (bf16) followed by glm_silu_mul_quant bit for bit on every live row,
    and leaves rows no expert owns untouched.  `wide` gives each row its own activation scale, 2^-30 .. 2^10,
    so the gate values run from below 2^-13 to above 2^7 (exp(-g) underflowing, overflowing and in range)."""
    T, n, k = 256, 512, 1024
    I = n // 2
    counts, psum, rows, a, sfa, w, sfb = grouped_case(T, n, k, seed=31)
    if wide:
        e = np.random.default_rng(32).integers(97, 138, rows).astype(np.uint8)
        v = sfa.reshape(-1, rows, 4)
        v[:] = e[None, :, None]
    da, dw, dsfa, dsfb, dpsum = d(a), d(w), d(sfa), d(sfb), d(psum)
    g13 = filled((rows, n), 0, torch.int16)
    ops.fp8_gemm_psum(da, dw, dsfa, dsfb, g13, dpsum, n=n, k=k, rows=rows, lda=k, ldc=n, sfa_rows=rows)
    tpad = torch.tensor([int((psum[-1] + 127) // 128 * 128)], dtype=torch.int32, device=DEV)
    q1 = filled((rows, I), 0x5c)
    sf1 = filled((ref.sf_words(I) * rows * 4,), 0x5d)
    ops.silu_mul_quant(g13, I, q1, sf1, rows, tpad, rows)
    q2 = filled((rows, I), 0x5c)
    sf2 = filled((ref.sf_words(I) * rows * 4,), 0x5d)
    ops.fp8_gemm_psum_silu_quant(da, dw, dsfa, dsfb, dpsum, q2, sf2, n=n, k=k, rows=rows, lda=k, sfa_rows=rows,
                                 sf_rows=rows)
    owned = np.zeros(rows, bool)
    for s0, s1 in ref.psum_ranges(psum):
        owned[s0:s1] = True
    Q1, Q2 = h(q1, np.uint8), h(q2, np.uint8)
    assert np.array_equal(Q1[owned], Q2[owned])
    assert np.all(Q2[~owned] == 0x5c)
    W1 = h(sf1, np.uint32).reshape(-1, rows)
    W2 = h(sf2, np.uint32).reshape(-1, rows)
    assert np.array_equal(W1[:, owned], W2[:, owned])
    assert np.all(W2[:, ~owned] == 0x5d5d5d5d)
    if wide:
        g = h(g13, np.uint16)[owned][:, :I]
        ex = (g >> 7) & 0xff
        assert (ex >= 134).any() and ((ex < 114) & ((g & 0x7fff) != 0)).any() and ((ex >= 114) & (ex < 134)).any()
        return
    # and against the oracle's chain: SiLU-mul-quant of bf16(the MFMA model's gate_up), every code and
    # exponent byte, where the model's gate_up equals the kernel's (>= 99.9% of the rows); the codes of the
    # fp32 reference's chain agree on > 97% (its bf16 gate_up differs in accumulation order)
    model = np.nan_to_num(ref.fp8_gemm_psum_mfma(a, w, sfa, sfb, psum, 256, n, k, rows, k, rows))
    g13_mod = ref.bf16_round(model)
    same = np.all(g13_mod == h(g13, np.uint16), axis=1) & owned
    assert same.sum() >= 0.999 * owned.sum()
    q3, sf3 = ref.silu_mul_quant(g13_mod, I, rows, None, rows,
                                 sf=np.full(ref.sf_words(I) * rows * 4, 0x5d, np.uint8))
    assert np.array_equal(q3[same], Q2[same])
    W3 = sf3.view(np.uint32).reshape(-1, rows)
    assert np.array_equal(W3[:, same], W2[:, same])
    ref32, _ = ref.fp8_gemm_psum(a, w, sfa, sfb, psum, 256, n, k, rows, k, rows)
    q4, _ = ref.silu_mul_quant(ref.bf16_round(np.nan_to_num(ref32.numpy())), I, rows, None, rows)
    print(f"PARITY fused gate_up codes: {np.mean(q4[owned] == Q2[owned]) * 100:.3f}% equal to the fp32 chain, "
          f"{same.sum()} of {owned.sum()} rows bit-exact against the MFMA-model chain", flush=True)
    assert np.mean(q4[owned] == Q2[owned]) > 0.97


# ------------------------------------------------------------------ bf16 batched (a4)

def bf16_ref_check(D_bits, A, B, k, what):
    ref32 = ref.bf16_batched(A.cpu(), B.cpu())
    S = ref.bf16_batched(A.cpu().float().abs().to(torch.float32), B.cpu().float().abs())
    out = torch.from_numpy(D_bits.view(np.int16)).view(torch.bfloat16).float()
    ok, rep = ref.check_bf16_gemm(out, ref32, S, k, steps_per_mfma=16)
    print(ref.parity_line(what, rep), flush=True)
    assert ok, ref.parity_line(what, rep)


def test_bf16_batched_uk_layout():
    """W_UK absorption as the reference lays it out (scripts/gen.py:136-137): A = qb[r][h*256 + 0:192],
    B = wuk[h][512][192], D = qmla[r][h][0:512] with columns 512-575 of every head untouched."""
    rows, m = 100, 97
    g = synth.generator(41)
    qb = (torch.randn(rows, 20480, generator=g)).to(torch.bfloat16).to(DEV)
    wuk = (torch.randn(64, 512, 192, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    qmla = filled((rows, 64, 576), SENTINEL, torch.int16)
    ops.bf16_batched(qb, wuk, qmla, m, n=512, k=192, rows=rows, a_strides=(40960, 512), b_strides=(384, 196608),
                     d_strides=(73728, 1152))
    D = h(qmla, np.uint16)
    A = qb[:m, :16384].view(m, 64, 256)[:, :, :192]
    bf16_ref_check(np.ascontiguousarray(D[:m, :, :512]), A, wuk, 192, "uk")
    assert np.all(D[:m, :, 512:] == SENTINEL) and np.all(D[m:] == SENTINEL)


def test_bf16_batched_uv_layout():
    """W_UV as the reference lays it out (scripts/gen.py:138-139, 401): A = o[r][h][512], B = kvb rows
    h*448 + 192 + d (a view offset 192*512 elements into kvb), D = ov[r][h][256]."""
    rows = 64
    g = synth.generator(42)
    o = torch.randn(rows, 64, 512, generator=g).to(torch.bfloat16).to(DEV)
    kvb = (torch.randn(64 * 448, 512, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    ov = filled((rows, 64, 256), SENTINEL, torch.int16)
    bview = kvb.view(-1)[192 * 512:]
    ops.bf16_batched(o, bview, ov, rows, n=256, k=512, rows=rows, a_strides=(65536, 1024), b_strides=(1024, 458752),
                     d_strides=(32768, 512))
    B = kvb.view(64, 448, 512)[:, 192:448, :]
    bf16_ref_check(h(ov, np.uint16), o, B, 512, "uv")


def test_bf16_batched_many_tiles():
    """Many tiles (1500 rows: 12 row tiles x 64 heads x 4 column tiles, more than the CUs hold at once) in the
    head-group tile order; M tail."""
    rows, m = 1504, 1500
    g = synth.generator(44)
    qb = (torch.randn(rows, 20480, generator=g)).to(torch.bfloat16).to(DEV)
    wuk = (torch.randn(64, 512, 192, generator=g) * 0.05).to(torch.bfloat16).to(DEV)
    qmla = filled((rows, 64, 576), SENTINEL, torch.int16)
    ops.bf16_batched(qb, wuk, qmla, m, n=512, k=192, rows=rows, a_strides=(40960, 512), b_strides=(384, 196608),
                     d_strides=(73728, 1152))
    D = h(qmla, np.uint16)
    A = qb[:m, :16384].view(m, 64, 256)[:, :, :192]
    bf16_ref_check(np.ascontiguousarray(D[:m, :, :512]), A, wuk, 192, "uk many tiles")
    assert np.all(D[:m, :, 512:] == SENTINEL) and np.all(D[m:] == SENTINEL)


def test_bf16_batched_bench_shapes_sampled():
    """W_UK and W_UV at the bench's 16384 rows in the reference's layouts; 8 rows of every head against the
    oracle."""
    M = 16384
    print("bf16 batched 16384 rows x 64 heads (W_UK, W_UV)", flush=True)
    g = synth.generator(45, "cuda")
    rows = sorted({0, 127, 128, M - 1} | set(np.random.default_rng(6).choice(M, 4, replace=False).tolist()))
    qb = torch.randn(M, 20480, generator=g, device=DEV).to(torch.bfloat16)
    wuk = (torch.randn(64, 512, 192, generator=g, device=DEV) * 0.05).to(torch.bfloat16)
    qmla = torch.empty(M, 64, 576, dtype=torch.bfloat16, device=DEV)
    ops.bf16_batched(qb, wuk, qmla, M, n=512, k=192, rows=M, a_strides=(40960, 512), b_strides=(384, 196608),
                     d_strides=(73728, 1152))
    A = qb[rows, :16384].view(len(rows), 64, 256)[:, :, :192].cpu()
    bf16_ref_check(h(qmla[rows, :, :512].contiguous().view(torch.int16), np.uint16), A, wuk.cpu(), 192, "uk 16384")
    del qb, qmla
    o = torch.randn(M, 64, 512, generator=g, device=DEV).to(torch.bfloat16)
    kvb = (torch.randn(64 * 448, 512, generator=g, device=DEV) * 0.05).to(torch.bfloat16)
    ov = torch.empty(M, 64, 256, dtype=torch.bfloat16, device=DEV)
    ops.bf16_batched(o, kvb.view(-1)[192 * 512:], ov, M, n=256, k=512, rows=M, a_strides=(65536, 1024),
                     b_strides=(1024, 458752), d_strides=(32768, 512))
    B = kvb.view(64, 448, 512)[:, 192:448, :].cpu()
    bf16_ref_check(h(ov[rows].contiguous().view(torch.int16), np.uint16), o[rows].cpu(), B, 512, "uv 16384")


def test_bf16_batched_k128_bench_shape_sampled():
    """W_UK in its contiguous K 128 form at full size: 64 heads x [16384 x 128] . [128 x 512] (the
    bench's aux.w_uk_k128_bf16_batched launch); tile-edge and random rows of every head against the oracle,
    every column, and the rows past m untouched."""
    M, rows = 16384, 16384 + 64
    print("bf16 batched 16384 rows x 64 heads, K 128", flush=True)
    g = synth.generator(46, "cuda")
    A = torch.randn(rows, 64, 128, generator=g, device=DEV).to(torch.bfloat16)
    B = (torch.randn(64, 512, 128, generator=g, device=DEV) * 0.1).to(torch.bfloat16)
    D = torch.full((rows, 64, 512), -3.0, dtype=torch.bfloat16, device=DEV)
    ops.bf16_batched(A, B, D, M, n=512, k=128, rows=rows, a_strides=(64 * 256, 256), b_strides=(256, 512 * 256),
                     d_strides=(64 * 1024, 1024))
    sample = sorted({0, 1, 127, 128, 255, 256, 8191, 8192, M - 2, M - 1} |
                    set(np.random.default_rng(7).choice(M, 8, replace=False).tolist()))
    bf16_ref_check(h(D[sample].contiguous().view(torch.int16), np.uint16), A[sample].cpu(), B.cpu(), 128,
                   f"k128 16384 ({len(sample)} rows)")
    assert bool((D[M:] == -3.0).all())


def test_bf16_batched_contiguous_k128():
    """The configured W_UK shape: 64 heads x [m x 128] . [128 x 512], contiguous operands, M tail."""
    rows, m = 130, 130
    g = synth.generator(43)
    A = torch.randn(rows, 64, 128, generator=g).to(torch.bfloat16).to(DEV)
    B = (torch.randn(64, 512, 128, generator=g) * 0.1).to(torch.bfloat16).to(DEV)
    D = filled((rows, 64, 512), SENTINEL, torch.int16)
    ops.bf16_batched(A, B, D, m, n=512, k=128, rows=rows, a_strides=(64 * 256, 256), b_strides=(256, 512 * 256),
                     d_strides=(64 * 1024, 1024))
    bf16_ref_check(h(D, np.uint16), A, B, 128, "k128")


# 64 heads and one head over the 256-column tiles of the batched kernel, with row and column tails
WIDE_BATCHED = [(64, 513, 264, 128)]
WIDE_F32 = [(33000, 264, 64, 272)]


@pytest.mark.parametrize("heads,m,n,k", WIDE_BATCHED)
def test_bf16_batched_wide_tiles_tail(heads, m, n, k):
    """Enough 128 x 256 tiles for the batched kernel to take them, their last column tile partial: against the oracle,
    nothing written past m and n."""
    print(f"bf16 batched {heads} heads {m} x {n} x {k}", flush=True)
    g = synth.generator(heads + m)
    A = torch.randn(m + 2, heads, k, generator=g).to(torch.bfloat16)
    B = (torch.randn(heads, n, k, generator=g) * 0.05).to(torch.bfloat16)
    D = filled((m + 2, heads, n + 8), SENTINEL, torch.int16)
    ops.bf16_batched(A.to(DEV), B.to(DEV), D, m, n=n, k=k, rows=m + 2, a_strides=(heads * k * 2, k * 2),
                     b_strides=(k * 2, n * k * 2), d_strides=(heads * (n + 8) * 2, (n + 8) * 2), heads=heads)
    out = h(D, np.uint16)
    bf16_ref_check(np.ascontiguousarray(out[:m, :, :n]), A[:m], B, k, f"wide {heads}x{m}x{n}x{k}")
    assert np.all(out[:m, :, n:] == SENTINEL) and np.all(out[m:] == SENTINEL)


@pytest.mark.parametrize("m,n,k,ldc", [(1000, 256, 6144, 256), (333, 32, 6144, 40), (16, 264, 192, 272),
                                       (40000, 256, 128, 256)] + WIDE_F32)
def test_gemm_f32_and_bf16(m, n, k, ldc):
    """The manifest's library GEMMs (scripts/gen.py:99-102): the MoE router's f32-output one (gen.py:435) and the
    indexer's bf16 weights_proj (gen.py:368), C = A . B^T; columns past n of each ldc row untouched."""
    g = synth.generator(m + n)
    A = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    B = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(DEV)
    ref32 = A.cpu().float() @ B.cpu().float().T
    S = A.cpu().float().abs() @ B.cpu().float().abs().T
    C32 = torch.full((m, ldc), -7.0, dtype=torch.float32, device=DEV)
    ops.gemm_f32(A, B, C32, m, n, k, ldc)
    got = C32.cpu()
    assert bool((got[:, n:] == -7.0).all())
    assert bool(((got[:, :n] - ref32).abs() <= (k / 16 + 32) * 2.0 ** -24 * S).all())
    C16 = filled((m, ldc), SENTINEL, torch.int16)
    ops.gemm_bf16(A, B, C16, m, n, k, ldc)
    D = h(C16, np.uint16)
    assert np.all(D[:, n:] == SENTINEL)
    out = torch.from_numpy(np.ascontiguousarray(D[:, :n]).view(np.int16)).view(torch.bfloat16).float()
    ok, rep = ref.check_bf16_gemm(out, ref32, S, k, steps_per_mfma=16)
    print(ref.parity_line(f"gemm_bf16 {m}x{n}x{k}", rep), flush=True)
    assert ok, ref.parity_line(f"gemm_bf16 {m}x{n}x{k}", rep)


# the 128 x 128 ring of the wide long-K library GEMMs: the bench's shape, and with row and column tails and an odd K
LIBRARY_128 = [(16384, 256, 6144, 256), (16001, 264, 1088, 272)]


@pytest.mark.parametrize("m,n,k,ldc", [(1000, 256, 6144, 264), (333, 32, 6144, 40), (130, 24, 1024, 24),
                                       (257, 72, 2048, 80), (64, 200, 1088, 208), (16384, 32, 6144, 32),
                                       (100, 64, 1216, 72), (77, 48, 3136, 56)] + LIBRARY_128)
def test_gemm_long_k_matches_batched(m, n, k, ldc):
    """Library GEMMs with K >= 1024 run the long-K kernels.  For n > 64 (rings of several stages, in 32 x 32, 64 x 64 or
    128 x 128 tiles by size) the bf16 outputs are the batched kernel's bit for bit (same MFMA chain over K; one head of kg_bf16_batched is the comparison); for
    n <= 64 (four K quarters summed in wave order) they are within the fp32 reference's accumulation bound.  bf16
    and f32 out, with row / column tails and columns past n of each ldc row untouched, and the f32 sums rounding
    to exactly the bf16 outputs (one set of sums, one rounding)."""
    g = synth.generator(7 * m + n)
    A = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    B = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(DEV)
    C32 = torch.full((m, ldc), -7.0, dtype=torch.float32, device=DEV)
    ops.gemm_f32(A, B, C32, m, n, k, ldc)
    C16 = filled((m, ldc), SENTINEL, torch.int16)
    ops.gemm_bf16(A, B, C16, m, n, k, ldc)
    D = h(C16, np.uint16)
    if n > 64:
        R16 = filled((m, 1, ldc), SENTINEL, torch.int16)
        ops.bf16_batched(A.view(m, 1, k), B.view(1, n, k), R16, m, n=n, k=k, rows=m, a_strides=(2 * k, 0),
                         b_strides=(2 * k, 0), d_strides=(2 * ldc, 0))
        R = h(R16, np.uint16).reshape(m, ldc)
        assert np.array_equal(D, R), f"bf16: {int((D != R).sum())} of {D.size} differ"
    else:
        assert np.all(D[:, n:] == SENTINEL)
        ref32 = A.cpu().float() @ B.cpu().float().T
        S = A.cpu().float().abs() @ B.cpu().float().abs().T
        out = torch.from_numpy(np.ascontiguousarray(D[:, :n]).view(np.int16)).view(torch.bfloat16).float()
        ok, rep = ref.check_bf16_gemm(out, ref32, S, k, steps_per_mfma=16)
        print(ref.parity_line(f"gemm_bf16 (K split) {m}x{n}x{k}", rep), flush=True)
        assert ok, ref.parity_line(f"gemm_bf16 (K split) {m}x{n}x{k}", rep)
        assert bool(((C32.cpu()[:, :n] - ref32).abs() <= (k / 16 + 32) * 2.0 ** -24 * S).all())
    got = C32.cpu()
    assert bool((got[:, n:] == -7.0).all())
    rb = got[:, :n].to(torch.bfloat16).view(torch.int16).numpy().view(np.uint16)
    assert np.array_equal(rb, D[:, :n])


LIBRARY_FEW = [(1, 72, 1024), (33, 264, 1088), (1300, 200, 1088), (2100, 264, 1984)]


@pytest.mark.parametrize("m,n,k", LIBRARY_FEW)
def test_gemm_few_rows_matches_batched(m, n, k):
    """The wide library GEMMs of few rows, in 32 x 32 and 64 x 64 tiles (by size) with row and column remainders and
    odd counts of 64-wide K steps: the bf16 outputs, and the f32 outputs rounded to bf16, are the batched kernel's bit
    for bit, and the f32 outputs are within the accumulation bound of the exact sums."""
    g = synth.generator(11 * m + n)
    A = torch.randn(m, k, generator=g).to(torch.bfloat16).to(DEV)
    B = (torch.randn(n, k, generator=g) * 0.02).to(torch.bfloat16).to(DEV)
    C32 = torch.full((m + 1, n + 8), -7.0, dtype=torch.float32, device=DEV)
    ops.gemm_f32(A, B, C32, m, n, k, n + 8)
    C16 = torch.full((m + 1, n + 8), -7.0, dtype=torch.bfloat16, device=DEV)
    ops.gemm_bf16(A, B, C16, m, n, k, n + 8)
    R16 = torch.empty(m, 1, n, dtype=torch.bfloat16, device=DEV)
    ops.bf16_batched(A.view(m, 1, k), B.view(1, n, k), R16, m, n=n, k=k, rows=m, a_strides=(2 * k, 0),
                     b_strides=(2 * k, 0), d_strides=(2 * n, 0))
    assert torch.equal(C16[:m, :n], R16[:, 0]) and torch.equal(C32[:m, :n].bfloat16(), R16[:, 0])
    ref64 = A.double() @ B.double().T
    S = A.double().abs() @ B.double().abs().T
    assert bool(((C32[:m, :n] - ref64).abs() <= (k / 16 + 32) * 2.0 ** -24 * S).all())
    assert bool((C32[:, n:] == -7).all()) and bool((C32[m:] == -7).all())
    assert bool((C16[:, n:] == -7).all()) and bool((C16[m:] == -7).all())


# ------------------------------------------------------------------ MQA logits (a5)

def mqa_case(num_q, num_kv, seed):
    g = synth.generator(seed)
    qf = torch.randn(num_q, 32, 128, generator=g).numpy()
    q8, qs = ref.head_quant(qf)
    kf = torch.randn(num_kv, 1, 128, generator=g).numpy()
    k8, ks_ = ref.head_quant(kf)
    k8 = k8.reshape(num_kv, 128)
    ksf = ks_.reshape(num_kv).astype(np.float32)
    iw = torch.randn(num_q, 32, generator=g).to(torch.bfloat16).float().numpy()
    w = (iw * qs * np.float32(0.08838834764831845) * np.float32(0.17677669529663687)).astype(np.float32)
    return q8, k8, ksf, w


def run_mqa(q8, k8, ksf, w, ks, ke, stride):
    num_q, num_kv = q8.shape[0], k8.shape[0]
    logits = filled((num_q, stride), -12345.0, torch.float32)
    ops.mqa_logits(d(q8), d(k8), d(ksf), d(w), d(ks.astype(np.uint32)), d(ke.astype(np.uint32)), logits, num_q,
                   num_kv, stride)
    return h(logits, np.float32)


def check_mqa(out, q8, k8, ksf, w, ks, ke, stride, what="mqa"):
    """Against the f64 reference: within the f32 summation bound plus the fp8 MFMA's own precision (2^-7 of each
    64-wide K group's largest product).  Against the oracle's model of the kernel's arithmetic (fp8 MFMA dots,
    its two head chains, then the key scale): at least 99.9% of the logits equal, the rest within 2^-20 of
    their |terms| sum (an MFMA output the model misses by an f32 ulp moves one head term).  Nothing is written
    past a row's key count."""
    num_q = q8.shape[0]
    want = ref.mqa_logits(q8, k8, ksf, w, ks, ke, num_q, stride).numpy()
    S = ref.mqa_logits_abs(q8, k8, ksf, w, ks, ke, num_q, stride).numpy()
    Wn = ref.mqa_logits_window(q8, k8, ksf, w, ks, ke, num_q, stride).numpy()
    model = ref.mqa_logits_mfma(q8, k8, ksf, w, ks, ke, num_q, stride)
    n_all = n_eq = 0
    worst = 0.0
    for r in range(num_q):
        n = int(ke[r] - ks[r])
        err = np.abs(out[r, :n] - want[r, :n])
        assert np.all(err <= 176 * 2.0 ** -24 * S[r, :n] + 2.0 ** -7 * Wn[r, :n] + 1e-30), f"row {r}: worst {err.max()}"
        assert np.all(out[r, n:] == -12345.0), f"row {r} written past its key count"
        dm = np.abs(out[r, :n].astype(np.float64) - model[r, :n])
        n_all += n
        n_eq += int((dm == 0).sum())
        if n:
            worst = max(worst, float((dm / (S[r, :n] + 1e-30)).max()))
    frac = n_eq / max(1, n_all)
    print(f"PARITY {what}: {n_eq} of {n_all} logits ({frac * 100:.4f}%) equal to the MFMA model, worst "
          f"|out - model| / sum|terms| {worst:.2e}", flush=True)
    assert frac >= 0.999 and worst <= 2.0 ** -20, (frac, worst)


def test_mqa_logits_bench_shape_sampled():
    """The bench's shape at full size: the last 16384 rows of one 65536-token sequence, causal, random e4m3
    codes and power-of-two key scales as the bench draws them; 6 rows (the first, the last, random) against
    the oracle over all their keys, and every row's tail past its key count untouched."""
    M, ctx = 16384, 65536
    print("mqa logits 16384 x 65536", flush=True)
    g = synth.generator(901, "cuda")
    codes = lambda *s: (torch.randint(0, 0x78, s, generator=g, device=DEV, dtype=torch.int32)
                        | (torch.randint(0, 2, s, generator=g, device=DEV, dtype=torch.int32) << 7)).to(torch.uint8)
    iq, kg = codes(M, 32, 128), codes(ctx, 128)
    ksf = torch.exp2(torch.randint(-8, 0, (ctx,), generator=g, device=DEV).float())
    w = torch.randn(M, 32, generator=g, device=DEV) * (128 ** -0.5) * (32 ** -0.5)
    ks = torch.zeros(M, dtype=torch.int32, device=DEV)
    ke = torch.arange(M, dtype=torch.int32, device=DEV) + (ctx - M) + 1
    logits = torch.full((M, ctx), -12345.0, dtype=torch.float32, device=DEV)
    ops.mqa_logits(iq, kg, ksf, w, ks, ke, logits, M, ctx, ctx)
    tail_ok = torch.arange(ctx, device=DEV)[None, :] < ke[:, None].long()
    assert bool(((logits == -12345.0) | tail_ok).all())                       # nothing written past ke
    rows = sorted({0, M - 1} | set(np.random.default_rng(5).choice(M, 4, replace=False).tolist()))
    out = h(logits[rows], np.float32)
    check_mqa(out, h(iq[rows], np.uint8), h(kg, np.uint8), h(ksf, np.float32), h(w[rows], np.float32),
              h(ks[rows], np.int32).astype(np.int64), h(ke[rows], np.int32).astype(np.int64), ctx)


def test_mqa_logits_ragged():
    num_q, num_kv, stride = 37, 1000, 1024
    q8, k8, ksf, w = mqa_case(num_q, num_kv, 51)
    rng = np.random.default_rng(52)
    ks = rng.integers(0, 500, num_q)
    ke = np.minimum(ks + rng.integers(0, 500, num_q), num_kv)
    ks[0], ke[0] = 10, 10            # an empty row
    ks[1], ke[1] = 0, num_kv         # every key
    ks[2], ke[2] = 999, 1000         # the last key only
    out = run_mqa(q8, k8, ksf, w, ks, ke, stride)
    check_mqa(out, q8, k8, ksf, w, ks, ke, stride)


@pytest.mark.parametrize("num_kv", [50, 64, 65, 129, 200, 320, 385])
def test_mqa_logits_short(num_kv):
    """Key ranges of one to seven 64-key blocks (the loop runs blocks in sixes after the first: the blocks past
    the last key store nothing)."""
    num_q, stride = 6, max(160, num_kv)
    q8, k8, ksf, w = mqa_case(num_q, num_kv, 55 + num_kv)
    rng = np.random.default_rng(num_kv)
    ks = rng.integers(0, num_kv, num_q)
    ke = np.minimum(ks + rng.integers(1, num_kv + 1, num_q), num_kv)
    out = run_mqa(q8, k8, ksf, w, ks, ke, stride)
    check_mqa(out, q8, k8, ksf, w, ks, ke, stride)


@pytest.mark.parametrize("num_q,num_kv", [(1, 447), (1, 448), (9, 449), (8, 897), (3, 2700), (17, 6000), (120, 3100)])
def test_mqa_logits_key_slices(num_q, num_kv):
    """Key ranges split over workgroups (slices of 7 or 13 blocks of 64 keys): ranges that end at, before and after
    a slice's edge, start inside one, and leave gaps between the rows of one workgroup."""
    print(f"mqa key slices {num_q} x {num_kv}", flush=True)
    q8, k8, ksf, w = mqa_case(num_q, num_kv, 77 + num_q)
    rng = np.random.default_rng(num_q)
    ks = np.zeros(num_q, np.int64)
    ke = np.full(num_q, num_kv) - np.arange(num_q)[::-1]
    if num_q > 2:
        ks[1::3] = num_kv - rng.integers(1, 200, len(ks[1::3]))       # the stream's end only
        ke[1::3] = num_kv
        ke[2::3] = rng.integers(0, 200, len(ke[2::3]))                # its start only (a gap between the two)
    out = run_mqa(q8, k8, ksf, w, ks, ke, (num_kv + 63) // 64 * 64)
    check_mqa(out, q8, k8, ksf, w, ks, ke, (num_kv + 63) // 64 * 64)


@pytest.mark.parametrize("num_q,seqs,ctx", [(5128, 20, 257), (5200, 9, 1100), (1030, 7, 513)])
def test_mqa_logits_straddling_groups(num_q, seqs, ctx):
    """Packed sequences whose edges fall inside groups of 8 rows, with fewer workgroups a group than the group's keys have
    slices (5128 and 5200 rows; longer slices) and with enough: each sequence's logits as in a call of its own."""
    print(f"mqa straddling {num_q} rows of {seqs}", flush=True)
    g = synth.generator(31, "cuda")
    codes = lambda *s: torch.randint(0, 0x78, s, generator=g, device=DEV, dtype=torch.uint8)
    iq, kg = codes(num_q, 32, 128), codes(seqs * ctx, 128)
    ksf = torch.exp2(torch.randint(-8, 0, (seqs * ctx,), generator=g, device=DEV).float())
    w = torch.randn(num_q, 32, generator=g, device=DEV)
    stride, row = (ctx + 255) // 256 * 256, 0
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    lens = [num_q // seqs + (i < num_q % seqs) for i in range(seqs)]
    ks = i32([i * ctx for i, n in enumerate(lens) for _ in range(n)])
    klen = i32([max(1, k) for n in lens for k in range(ctx - n + 1, ctx + 1)])
    out = torch.full((num_q, stride), -12345.0, device=DEV)
    ops.mqa_logits(iq, kg, ksf, w, ks, ks + klen, out, num_q, seqs * ctx, stride)
    for i, n in enumerate(lens):
        own, sl, keys = torch.full((n, stride), -12345.0, device=DEV), slice(row, row + n), slice(i * ctx, (i + 1) * ctx)
        ops.mqa_logits(iq[sl], kg[keys], ksf[keys].clone(), w[sl].clone(), torch.zeros_like(klen[sl]), klen[sl].clone(), own,
                       n, ctx, stride)
        assert torch.equal(out[sl], own), f"sequence {i}"
        row += n


@pytest.mark.parametrize("num_q,seqs,ctx", [(13814, 20, 691), (1024, 64, 1024)])
def test_mqa_logits_packed_time(num_q, seqs, ctx):
    """Many short sequences take about the time of the same rows with the same key counts over one sequence's keys: no
    workgroups for the other sequences' keys (which took 2.1 and 1.8 times it)."""
    g = synth.generator(21, "cuda")
    codes = lambda *s: torch.randint(0, 0x78, s, generator=g, device=DEV, dtype=torch.uint8)
    iq, kg = codes(num_q, 32, 128), codes(seqs * ctx, 128)
    ksf, w = torch.ones(seqs * ctx, device=DEV), torch.randn(num_q, 32, generator=g, device=DEV)
    lens = [num_q // seqs + (i < num_q % seqs) for i in range(seqs)]
    ks = torch.tensor([i * ctx for i, n in enumerate(lens) for _ in range(n)], dtype=torch.int32, device=DEV)
    klen = torch.tensor([k for n in lens for k in range(ctx - n + 1, ctx + 1)], dtype=torch.int32, device=DEV)
    stride = (ctx + 255) // 256 * 256
    logits = torch.empty(num_q, stride, dtype=torch.float32, device=DEV)
    zero, ke = torch.zeros_like(ks), ks + klen
    one, packed = fastest([lambda: ops.mqa_logits(iq, kg, ksf, w, zero, klen, logits, num_q, ctx, stride),
                           lambda: ops.mqa_logits(iq, kg, ksf, w, ks, ke, logits, num_q, seqs * ctx, stride)])
    print(f"mqa {num_q} rows: one sequence {one:.1f} us, {seqs} sequences {packed:.1f}", flush=True)
    assert packed <= 1.4 * one


def test_mqa_logits_causal_chunk():
    """The benchmark's shape at reduced size: the last 256 rows of one 4096-token sequence, causal."""
    num_q, num_kv, stride = 256, 4096, 4096
    q8, k8, ksf, w = mqa_case(num_q, num_kv, 53)
    ks = np.zeros(num_q, np.int64)
    ke = np.arange(num_kv - num_q, num_kv) + 1
    out = run_mqa(q8, k8, ksf, w, ks, ke, stride)
    check_mqa(out, q8, k8, ksf, w, ks, ke, stride)


def test_mqa_logits_packed_sequences():
    """Rows of three packed sequences: each row scores its own sequence's keys [goff, goff + pos + 1)."""
    lens = [300, 1, 700]
    goff = np.cumsum([0] + lens[:-1])
    ks, ke = [], []
    for s, L in enumerate(lens):
        for p in range(max(0, L - 40), L):          # the chunk holds each sequence's last (up to) 40 rows
            ks.append(goff[s])
            ke.append(goff[s] + p + 1)
    ks, ke = np.array(ks), np.array(ke)
    num_q, num_kv, stride = len(ks), sum(lens), 768
    q8, k8, ksf, w = mqa_case(num_q, num_kv, 54)
    out = run_mqa(q8, k8, ksf, w, ks, ke, stride)
    check_mqa(out, q8, k8, ksf, w, ks, ke, stride)
