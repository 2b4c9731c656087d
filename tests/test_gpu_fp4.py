"""GPU parity of the FP4 decode kernels against the CPU oracle: FP16 bits
bit-exact, and the reference's ValueError conditions raised in its order."""
import numpy as np
import pytest
import torch

import cases

pytestmark = pytest.mark.gpu


def g16_packet(rng, rows, cols, device, *, global_scale=None):
    """Random nibbles; block scales per the BASELINE recipe: s ~ lognormal(-3,
    0.5), global = max(s)/448, block byte = E4M3(clamp(s/global, 0, 448))."""
    groups = (cols + 15) // 16
    packed = rng.integers(0, 256, size=(rows, groups * 8), dtype=np.uint16).astype(np.uint8)
    if cols % 16:
        # zero the padding nibbles of the final group
        codes = np.stack((packed & 15, packed >> 4), -1).reshape(rows, -1)
        codes[:, cols:] = 0
        packed = (codes[:, 0::2] | (codes[:, 1::2] << 4)).astype(np.uint8)
    s = np.exp(rng.normal(-3.0, 0.5, size=(rows, groups))).astype(np.float32)
    g = np.float32(s.max() / 448.0) if global_scale is None else np.float32(global_scale)
    sb = torch.from_numpy(np.clip(s / g, 0, 448)).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    return packed, sb, g


def decode_dev(packed, scales_u8, g, rows, cols, device, group=16):
    from mamba2_recall import fp4
    pk = torch.from_numpy(packed).to(device)
    if group == 16:
        sc = torch.from_numpy(scales_u8).to(device).view(torch.float8_e4m3fn)
        packet = dict(format="fp4_g16_e4m3", shape=[rows, cols], group_size=16, packed=pk, scales=sc,
                      global_scale=torch.tensor(g, dtype=torch.float32))
    else:
        sc = torch.from_numpy(scales_u8.view(np.float16)).to(device)
        packet = dict(format="fp4_g64_f16", shape=[rows, cols], group_size=64, packed=pk, scales=sc,
                      global_scale=None)
    return fp4.decode_packet(packet)


# (33, 4112): 16 whole blocks of 1024 units for the wide-load kernel and 578 units for the per-unit one
@pytest.mark.parametrize("rows,cols", [(512, 4096), (37, 8192), (33, 4112), (3, 48), (5, 40)])
def test_g16_random_bit_exact(oracle, device, rows, cols):
    rng = np.random.default_rng(rows * 7 + cols)
    packed, sb, g = g16_packet(rng, rows, cols, device)
    print(f"[fp4 g16] rows={rows} cols={cols}", flush=True)
    want, err = oracle.fp4_decode(16, packed, sb, g, rows, cols)
    assert err == 0
    got = decode_dev(packed, sb, g, rows, cols, device).cpu().numpy().view(np.uint16)
    assert int((got != want).sum()) == 0


def test_g16_every_code_every_scale_byte(oracle, device):
    """All 16 codes x all 254 finite non-negative-or-zero scale bytes x a set
    of globals, including ones that overflow FP16 (must raise)."""
    scale_bytes = np.array([b for b in range(256) if (b & 0x7F) != 0x7F and (b < 0x80 or b == 0x80)], np.uint8)
    codes = np.arange(16, dtype=np.uint8)
    for g in (1.0, 2.0 ** -20, 0.3, 1.7e-3, 100.0, 2.0 ** 24):
        rows = scale_bytes.size
        cols = 16 * 16
        code_mat = np.tile(np.repeat(codes, 16), (rows, 1))              # group j holds code j
        sb = np.repeat(scale_bytes[:, None], 16, axis=1)                  # [rows, 16 groups]
        # zero scale bytes may only hold codes 0/8: keep those rows' other groups at code 0
        zero_rows = (scale_bytes & 0x7F) == 0
        code_mat[zero_rows] = np.where(np.isin(code_mat[zero_rows], (0, 8)), code_mat[zero_rows], 0)
        packed = (code_mat[:, 0::2] | (code_mat[:, 1::2] << 4)).astype(np.uint8)
        want, err = oracle.fp4_decode(16, packed, sb, g, rows, cols)
        print(f"[fp4 g16 KAT] global={g} err={err}", flush=True)
        if err:
            assert err == 8, err
            with pytest.raises(ValueError, match="Nonfinite decoded FP16 weights"):
                decode_dev(packed, sb, g, rows, cols, device)
            continue
        got = decode_dev(packed, sb, g, rows, cols, device).cpu().numpy().view(np.uint16)
        assert int((got != want).sum()) == 0
        # closed form: FP16(FP32(FP32(lev*sign*block)*global)) via numpy float32
        lev = np.array([0, .5, 1, 1.5, 2, 3, 4, 6], np.float32)
        blk = torch.from_numpy(sb).view(torch.float8_e4m3fn).float().numpy()
        c = code_mat.reshape(rows, 16, 16)
        val = (lev[c & 7] * np.where(c & 8, np.float32(-1), np.float32(1))).astype(np.float32)
        val = (val * blk[:, :, None]).astype(np.float32) * np.float32(g)
        closed = val.astype(np.float32).astype(np.float16).view(np.uint16).reshape(rows, cols)
        assert int((closed != got).sum()) == 0


def _assert_equal_in_chunks(got_dev, want, rows_per_chunk=16384):
    for r0 in range(0, want.shape[0], rows_per_chunk):
        got = got_dev[r0:r0 + rows_per_chunk].cpu().numpy().view(np.uint16)
        bad = int((got != want[r0:r0 + rows_per_chunk]).sum())
        assert bad == 0, f"rows {r0}..: {bad} mismatched FP16 weights"


def test_g16_embedding_matrix_bit_exact(oracle, device):
    """The [256000, 4096] embedding / lm_head matrix of the full 8B set
    (131,072,000 eight-weight units) at the automatic decode shape: one pass
    of 128,000 workgroups."""
    rows, cols = 256000, 4096
    rng = np.random.default_rng(256000)
    packed = rng.integers(0, 256, size=(rows, cols // 2), dtype=np.uint8)
    s = np.exp(rng.normal(-3.0, 0.5, size=(rows, cols // 16))).astype(np.float32)
    g = np.float32(s.max() / 448.0)
    sb = torch.from_numpy(np.clip(s / g, 0, 448)).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    del s
    print(f"[fp4 g16 embedding] rows={rows} cols={cols} units={rows * cols // 8}", flush=True)
    want, err = oracle.fp4_decode(16, packed, sb, g, rows, cols)
    assert err == 0
    _assert_equal_in_chunks(decode_dev(packed, sb, g, rows, cols, device), want)


def _forced_fp4_shape(upt, cap, nt):
    from mamba2_recall import _native
    lib = _native.lib()
    assert lib.m2r_set_fp4_decode_shape(upt, cap, nt) == 0
    return lib


@pytest.mark.parametrize("upt,cap,nt", [(1, 2048, 1), (2, 4096, 0), (4, 2048, 1), (4, 0, 0), (8, 1024, 0),
                                        (8, 0, 1)])
def test_g16_forced_shapes_and_grid_stride_sweeps(oracle, device, upt, cap, nt):
    """Every decode shape the tuning hook offers gives the oracle's weights:
    1-8 units per thread, default and non-temporal stores, and grid caps of
    1024-4096 workgroups, which make each workgroup stride over the
    [4096, 8192] out_proj matrix (4,194,304 units) in 2 to 16 sweeps."""
    rows, cols = 4096, 8192
    rng = np.random.default_rng(upt * 100 + cap + nt)
    packed = rng.integers(0, 256, size=(rows, cols // 2), dtype=np.uint8)
    s = np.exp(rng.normal(-3.0, 0.5, size=(rows, cols // 16))).astype(np.float32)
    g = np.float32(s.max() / 448.0)
    sb = torch.from_numpy(np.clip(s / g, 0, 448)).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    print(f"[fp4 g16 shape] upt={upt} cap={cap} nt={nt}", flush=True)
    want, err = oracle.fp4_decode(16, packed, sb, g, rows, cols)
    assert err == 0
    lib = _forced_fp4_shape(upt, cap, nt)
    try:
        got = decode_dev(packed, sb, g, rows, cols, device)
    finally:
        lib.m2r_set_fp4_decode_shape(0, 0, 1)
    _assert_equal_in_chunks(got, want)


def test_g64_grid_stride_sweeps(oracle, device):
    """G64 under a forced grid cap of 2048 workgroups: 20,480,000 units in
    ten sweeps."""
    rows, cols = 40000, 4096
    rng = np.random.default_rng(40000)
    packed = rng.integers(0, 256, size=(rows, cols // 2), dtype=np.uint8)
    sc = np.exp(rng.normal(-3.0, 0.5, size=(rows, cols // 64))).astype(np.float16).view(np.uint16)
    print(f"[fp4 g64 sweeps] rows={rows} cols={cols} units={rows * cols // 8}", flush=True)
    want, err = oracle.fp4_decode(64, packed, sc, 1.0, rows, cols)
    assert err == 0
    lib = _forced_fp4_shape(4, 2048, 1)
    try:
        got = decode_dev(packed, sc, None, rows, cols, device, group=64)
    finally:
        lib.m2r_set_fp4_decode_shape(0, 0, 1)
    _assert_equal_in_chunks(got, want)
    _assert_equal_in_chunks(decode_dev(packed, sc, None, rows, cols, device, group=64), want)


# (19, 8256): 19 whole blocks of 1024 units for the wide-load kernel and 152 units for the per-unit one
@pytest.mark.parametrize("rows,cols", [(64, 4096), (19, 8256), (7, 192), (3, 100)])
def test_g64_random_bit_exact(oracle, device, rows, cols):
    rng = np.random.default_rng(rows + cols)
    groups = (cols + 63) // 64
    codes = rng.integers(0, 16, size=(rows, groups * 64)).astype(np.uint8)
    codes[:, cols:] = 0
    packed = (codes[:, 0::2] | (codes[:, 1::2] << 4)).astype(np.uint8)
    sc = np.exp(rng.normal(-3.0, 0.5, size=(rows, groups))).astype(np.float16).view(np.uint16)
    print(f"[fp4 g64] rows={rows} cols={cols}", flush=True)
    want, err = oracle.fp4_decode(64, packed, sc, 1.0, rows, cols)
    assert err == 0
    got = decode_dev(packed, sc, None, rows, cols, device, group=64).cpu().numpy().view(np.uint16)
    assert int((got != want).sum()) == 0


@pytest.mark.parametrize("group", [16, 64])
@pytest.mark.parametrize("rows,cols", [(3, 8), (5, 9), (2, 15), (7, 17), (67, 31), (1000, 33), (129, 63), (5, 65),
                                       (3, 2730), (3, 2731), (9, 4100), (2, 8191), (3, 8193), (1, 20001), (4, 7),
                                       (131080, 8), (120001, 9), (87400, 12)])
def test_ragged_widths_bit_exact(oracle, device, group, rows, cols):
    """Widths that are no multiple of the group: rows and groups that end
    anywhere in an eight-weight vector, a partial last vector, widths on both
    sides of a workgroup's 8192 weights, one below eight columns, and short
    rows on both sides of 2^20 weights."""
    if cols % group == 0:
        return
    rng = np.random.default_rng(rows * 31 + cols + group)
    groups = (cols + group - 1) // group
    codes = rng.integers(0, 16, size=(rows, groups * group)).astype(np.uint8)
    codes[:, cols:] = 0
    packed = (codes[:, 0::2] | (codes[:, 1::2] << 4)).astype(np.uint8)
    s = np.exp(rng.normal(-3.0, 0.5, size=(rows, groups))).astype(np.float32)
    g = np.float32(s.max() / 448.0)
    if group == 16:
        sc = torch.from_numpy(np.clip(s / g, 0, 448)).to(torch.float8_e4m3fn).view(torch.uint8).numpy()
    else:
        sc, g = s.astype(np.float16).view(np.uint16), None
    print(f"[fp4 ragged] group={group} rows={rows} cols={cols}", flush=True)
    want, err = oracle.fp4_decode(group, packed, sc, 1.0 if g is None else g, rows, cols)
    assert err == 0
    got = decode_dev(packed, sc, g, rows, cols, device, group=group).cpu().numpy().view(np.uint16)
    assert int((got != want).sum()) == 0
    if rows > 2:   # the error bits, in the middle and at the ends
        for r, c in ((0, cols - 1), (rows // 2, 0), (rows - 1, cols // 2), (rows - 1, cols - 1)):
            bad = sc.copy()
            bad[r, c // group] = 0
            pk = packed.copy()
            pk[r, c // 2] = 0x11 & (0x0F if cols % 2 and c == cols - 1 else 0xFF)
            with pytest.raises(ValueError, match="Nonzero code in a zero-scale group"):
                decode_dev(pk, bad, g, rows, cols, device, group=group)
            bad[r, c // group] = 0x7F if group == 16 else 0x7E00
            with pytest.raises(ValueError, match="Invalid stored scale"):
                decode_dev(packed, bad, g, rows, cols, device, group=group)
        for r, c in ((0, cols), (rows - 1, groups * group - 1), (rows // 2, cols)):
            pk = packed.copy()
            pk[r, c // 2] |= 0x10 if c % 2 else 0x01
            with pytest.raises(ValueError, match="Nonzero final-group padding"):
                decode_dev(pk, sc, g, rows, cols, device, group=group)


def test_decode_errors_follow_reference_order(device):
    rng = np.random.default_rng(5)
    rows, cols = 4, 64
    packed, sb, g = g16_packet(rng, rows, cols, device)
    bad = sb.copy(); bad[1, 2] = 0x7F                        # NaN block scale
    with pytest.raises(ValueError, match="Invalid stored scale"):
        decode_dev(packed, bad, g, rows, cols, device)
    bad = sb.copy(); bad[0, 0] = 0xB8                        # negative block scale
    with pytest.raises(ValueError, match="Invalid stored scale"):
        decode_dev(packed, bad, g, rows, cols, device)
    with pytest.raises(ValueError, match="Global scale must be finite and positive"):
        decode_dev(packed, sb, 0.0, rows, cols, device)
    bad = sb.copy(); bad[2, 1] = 0x00                        # zero block with nonzero codes
    pk = packed.copy(); pk[2, 8:16] = 0x31
    with pytest.raises(ValueError, match="Nonzero code in a zero-scale group"):
        decode_dev(pk, bad, g, rows, cols, device)
    pk = packed.copy(); pk[2, 8:16] = 0x88                   # codes 8 (= -0) are allowed
    out = decode_dev(pk, bad, g, rows, cols, device).cpu().numpy().view(np.uint16)
    assert (out[2, 16:32] == 0x8000).all()
    p2, s2, g2 = g16_packet(rng, 2, 40, device)
    p2[:, -1] |= 0x30                                         # padding nibble (column 41) nonzero
    with pytest.raises(ValueError, match="Nonzero final-group padding"):
        decode_dev(p2, s2, g2, 2, 40, device)


@pytest.mark.parametrize("M,N,K", [(1, 18560, 4096), (2, 1000, 4096), (4, 333, 4096), (1, 4096, 8192),
                                   (2, 257, 8192), (4, 101, 8192), (1, 100, 2048), (4, 63, 2048), (1, 1, 4096)])
def test_fp4_gemv_matches_decoded_weights(device, M, N, K):
    """fp4.gemv_g16 (packed-resident FP4 G16 GEMV) against the product with
    the decoded FP16 weights (decode_packet, bit-exact to the oracle) in
    float64: relative L2 <= 1e-3 (north_star tolerance), and every output
    within one binary16 ulp plus the binary32 accumulation bound K * 2^-22 *
    sum|u w|.  Packets in the reference G16 format, with some zero-scale
    groups holding codes 0 and 8."""
    import torch
    from mamba2_recall import fp4
    gen = torch.Generator(device=device).manual_seed(M * 7919 + N)
    print(f"[fp4 gemv] M={M} N={N} K={K}", flush=True)
    packed = torch.randint(0, 256, (N, K // 2), generator=gen, device=device, dtype=torch.uint8)
    s = torch.exp(torch.randn((N, K // 16), generator=gen, device=device) * 0.5 - 3.0)
    g = (s.max() / 448.0).float().reshape(1)
    sb = (s / g).clamp(0, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    zero = torch.rand((N, K // 16), generator=gen, device=device) < 0.02
    sb = torch.where(zero, torch.zeros_like(sb), sb)
    codes = packed.view(N, K // 16, 8)
    codes = torch.where(zero[..., None], codes & 0x88, codes).view(N, K // 2)
    w = fp4.decode_packet(dict(format="fp4_g16_e4m3", shape=[N, K], group_size=16, packed=codes,
                               scales=sb.view(torch.float8_e4m3fn), global_scale=g.reshape(())))
    u = torch.randn((M, K), generator=gen, device=device).half()
    y = fp4.gemv_g16(codes, sb, g, u)
    ref = u.double() @ w.double().T
    torch.cuda.synchronize()
    err = (y.double() - ref).norm() / ref.norm()
    assert float(err) <= 1e-3, float(err)
    bound = (ref.abs() * 2.0 ** -11 + (u.double().abs() @ w.double().abs().T) * K * 2.0 ** -22 + 2.0 ** -24)
    assert bool(((y.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("N,K,tiny", [(1, 2048, 1.0), (16, 2048, 1.0), (17, 2048, 1.0), (2033, 8192, 1.0),
                                      (2048, 4096, 1.0), (4111, 4096, 1.0), (40003, 2048, 1.0),
                                      (5000, 8192, 2.0 ** -16)])
def test_fp4_gemv_four_rows_tiles(device, N, K, tiny):
    """The matrix-core GEMV (four activation rows) around its 16-row tiles and
    its batches of eight tiles per workgroup (N > 32,768), and with weights
    down to binary16 subnormals, against float64 within the bounds of the test
    above: products of binary16 values are exact in binary32.  Then with
    weights that are multiples of 1/2 up to 24 and whole activations up to 8:
    every sum is exact in binary32 (below 2^23 halves), so the outputs must
    equal the product, and a lost or misplaced code word shows."""
    from mamba2_recall import fp4
    gen = torch.Generator(device=device).manual_seed(N + K)
    print(f"[fp4 gemv tiles] N={N} K={K} tiny={tiny}", flush=True)
    codes = torch.randint(0, 256, (N, K // 2), generator=gen, device=device, dtype=torch.uint8)
    s = torch.exp(torch.randn((N, K // 16), generator=gen, device=device) * 0.5 - 3.0)
    g = (s.max() / 448.0).float().reshape(1)
    sb = (s / g).clamp(0, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    sb = torch.where(sb == 0, torch.ones_like(sb), sb)
    g = g * tiny
    w = fp4.decode_packet(dict(format="fp4_g16_e4m3", shape=[N, K], group_size=16, packed=codes,
                               scales=sb.view(torch.float8_e4m3fn), global_scale=g.reshape(())))
    if tiny < 1:
        assert float((w.abs().float() < 2.0 ** -14).float().mean()) > 0.5
    wide = torch.randn((4, K + 8), generator=gen, device=device).half()
    for u in (wide[:, :K].contiguous(), wide[:, :K]):   # the second with a row stride of its own
        y = fp4.gemv_g16(codes, sb, g, u)
        ref = u.double() @ w.double().T
        assert float((y.double() - ref).norm() / ref.norm()) <= (1e-3 if tiny == 1.0 else 1e-2)   # (subnormal outputs)
        bound = (ref.abs() * 2.0 ** -11 + (u.double().abs() @ w.double().abs().T) * K * 2.0 ** -22 + 2.0 ** -24)
        assert bool(((y.double() - ref).abs() <= bound).all())
    whole = torch.tensor([0x38, 0x40, 0x48], device=device, dtype=torch.uint8)   # block scales 1, 2 and 4
    sb = whole[torch.randint(0, 3, (N, K // 16), generator=gen, device=device)]
    one = torch.ones(1, device=device)
    w = fp4.decode_packet(dict(format="fp4_g16_e4m3", shape=[N, K], group_size=16, packed=codes,
                               scales=sb.view(torch.float8_e4m3fn), global_scale=one.reshape(())))
    u = torch.randint(-8, 9, (4, K), generator=gen, device=device).half()
    assert torch.equal(fp4.gemv_g16(codes, sb, one, u), (u.double() @ w.double().T).half())


@pytest.mark.parametrize("N,K", [(1, 4096), (100, 8192), (1500, 4096), (2032, 8192)])
def test_fp4_gemv_four_rows_of_few_outputs_same_bits(device, N, K):
    """Outputs that give fewer than half the CUs a tile stay with the dot
    products: four activation rows have the bits of two times two."""
    from mamba2_recall import fp4
    if torch.cuda.get_device_properties(device).multi_processor_count != 256:
        pytest.skip("the line lies at half of 256 CUs")
    gen = torch.Generator(device=device).manual_seed(N + K)
    print(f"[fp4 gemv four rows, few outputs] N={N} K={K}", flush=True)
    codes = torch.randint(0, 256, (N, K // 2), generator=gen, device=device, dtype=torch.uint8)
    sb = torch.randint(40, 90, (N, K // 16), generator=gen, device=device, dtype=torch.uint8)
    g = torch.full((1,), 0.003, device=device)
    u = torch.randn((4, K), generator=gen, device=device).half()
    four = fp4.gemv_g16(codes, sb, g, u)
    two = torch.cat([fp4.gemv_g16(codes, sb, g, u[i:i + 2]) for i in (0, 2)])
    assert torch.equal(four.view(torch.int16), two.view(torch.int16))


@pytest.mark.parametrize("N,K", [(18560, 4096), (4640, 4096), (4096, 8192), (2048, 8192), (100, 2048)])
def test_fp4_gemv_one_row_same_bits_as_two_rows(device, N, K):
    """One activation row runs the whole-row kernel where it fills the chip in
    one resident round (in_proj and out_proj shapes of the 8B model), several
    rows the general kernel; both add each row's 2048-wide chunk sums (wave
    sums) in chunk order, so y of one row equals row 0 of the same row passed
    twice, bit for bit."""
    from mamba2_recall import fp4
    gen = torch.Generator(device=device).manual_seed(N + K)
    print(f"[fp4 gemv one row] N={N} K={K}", flush=True)
    codes = torch.randint(0, 256, (N, K // 2), generator=gen, device=device, dtype=torch.uint8)
    s = torch.exp(torch.randn((N, K // 16), generator=gen, device=device) * 0.5 - 3.0)
    g = (s.max() / 448.0).float().reshape(1)
    sb = (s / g).clamp(0, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    u = torch.randn((1, K), generator=gen, device=device).half()
    y1 = fp4.gemv_g16(codes, sb, g, u)
    y2 = fp4.gemv_g16(codes, sb, g, torch.cat((u, u)))
    torch.cuda.synchronize()
    assert torch.equal(y1[0].view(torch.int16), y2[0].view(torch.int16))
    assert torch.equal(y2[0].view(torch.int16), y2[1].view(torch.int16))
