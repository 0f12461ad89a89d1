"""The prefill kernel (csrc/prefill_q.hip) at the edges of its tiles: token and
row remainders, partial super-steps of K, every tile and K split its plan picks,
one and three activation terms, the GLU epilogue's bits, and the scratch it
keeps between calls."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _say(msg):
    print(f"\n[prefill] {msg}", flush=True)


def _weight(orc, dev, N, K, seed):
    """A registered projection and its dequantized matrix in float64 (the
    dequantization itself is pinned bit for bit by test_gpu_parity.py)."""
    import alveare_amd as aa

    W = torch.from_numpy(orc.synth_q4(N, K, seed)).to(dev)
    return aa.Q4Weight(W, N, K), aa.dequant_q4(W, N, K).double()


def _plan(M, N, K, fp32=False, ffn=0):
    """(tokens per workgroup, K splits) of the prefill kernel, (0, 0) for the
    LDS tile kernel of csrc/gemm_q.hip."""
    import ctypes

    import alveare_amd as aa

    t, k = ctypes.c_int(), ctypes.c_int()
    aa._lib.check(aa.lib().alv_prefill_plan(M, N, K, int(fp32), ffn, ctypes.byref(t), ctypes.byref(k)), "plan")
    return t.value, k.value


# M, N, K and the plan of a 256-CU card: every tile, unsplit and at splits the
# plan takes, token and row remainders, whole (1984) and partial super-steps; then
# the LDS tile kernel on registered weights, 64- and 256-token tiles.
PRODUCTS = {
    "bf16": [(18, 69, 576, 32, 1), (130, 333, 480, 32, 1), (21, 67, 1984, 32, 2), (138, 67, 4000, 32, 4),
             (18, 69, 16064, 32, 8), (19, 69, 16288, 32, 16), (98, 20247, 544, 64, 1), (33, 23714, 1984, 64, 2),
             (2849, 131, 4000, 64, 4), (33, 6369, 8128, 64, 8), (290, 19501, 544, 128, 1), (68, 31169, 3424, 128, 2),
             (71, 16299, 5920, 128, 4), (265, 29911, 544, 192, 1), (132, 28098, 3648, 192, 2), (129, 15296, 7456, 192, 4),
             (775, 13825, 544, 256, 1),
             (17, 333, 480, 0, 0), (31, 1000, 32, 0, 0), (64, 8192, 3840, 0, 0), (1000, 1111, 96, 0, 0),
             (3000, 1536, 1152, 0, 0),
             (600, 2000, 3872, 64, 2), (70, 512, 15360, 0, 0), (600, 544, 15360, 64, 8),
             (193, 30001, 544, 0, 0), (300, 30720, 1024, 192, 1), (490, 30000, 1056, 256, 1)],
    "fp32": [(34, 96, 1984, 32, 2), (37, 69, 5152, 32, 4), (36, 96, 16288, 32, 16), (70, 28608, 96, 64, 1),
             (34, 10048, 4160, 64, 4), (67, 21920, 2336, 128, 2), (69, 8128, 8160, 128, 8), (276, 22304, 544, 192, 1),
             (131, 7008, 8352, 192, 8), (390, 22112, 576, 256, 1), (206, 25152, 6048, 256, 2),
             (33, 333, 64, 0, 0), (700, 9000, 160, 0, 0),
             (600, 2000, 3872, 64, 2), (70, 512, 15360, 32, 8), (600, 544, 15360, 64, 8),
             (193, 30001, 544, 128, 1), (300, 30720, 1024, 192, 1), (490, 30000, 1056, 256, 1)],
}


# (fp32 activations take the streaming kernel below 33 tokens)
@pytest.mark.parametrize("M,N,K,tokens,splits,dtype", [(*s, d) for d, shapes in PRODUCTS.items() for s in shapes])
def test_prefill_products(orc, dev, M, N, K, tokens, splits, dtype):
    """Within the float32 bound of the float64 product: K + 8 roundings of 2^-24
    over sum |x w| (three terms: 3 K + 8), a bf16 result half a bf16 ulp more
    (2^-8 of the value: eight significant bits)."""
    from alveare_amd import layer

    _say(f"product M={M} N={N} K={K} {dtype}")
    assert _plan(M, N, K, dtype == "fp32") == (tokens, splits)
    w, w64 = _weight(orc, dev, N, K, M + N)
    x = torch.from_numpy(orc.synth_normal(M * K, M + K)).to(dev).view(M, K)
    x = x.to(torch.bfloat16) if dtype == "bf16" else x
    y = layer.gemv_bf16(w, x, M=M).view(M, N) if dtype == "bf16" else w(x, M=M)
    x64 = x.double()
    ref = x64 @ w64.T
    bound = ((3 if dtype == "fp32" else 1) * K + 8) * 2.0 ** -24 * (x64.abs() @ w64.abs().T) + 1e-30
    if dtype == "bf16":
        bound = bound * 1.01 + ref.abs() * 2.0 ** -8
    bad = ((y.double() - ref).abs() > bound).sum().item()
    assert bad == 0, f"{bad} of {M * N} outside the float32 bound"
    w.close()


def _picker(I, H, cols):
    """Combined-layout rows whose only nonzero weight is 1 at column cols[i]."""
    W = np.zeros((I, H // 32, 20), np.uint8)
    W[:, :, 17] = 0x3F  # bf16 1.0
    W[:, :, 16] = 0x80
    c = np.asarray(cols)
    W[np.arange(I), c // 32, (c % 32) // 2] = np.where(c % 2, 0x10, 0x01)
    return W.reshape(I, -1)


# M, I, H (the K of gate/up) and its plan: every tile, unsplit and split.
GLU = [(480, 15360, 1056, 256, 1), (17, 2080, 1056, 32, 1), (330, 2080, 1056, 32, 1), (17, 96, 1984, 32, 2),
       (26, 64, 4000, 32, 4), (65, 13152, 544, 64, 1), (33, 10176, 2176, 64, 2), (33, 5440, 4032, 64, 4),
       (33, 3008, 8608, 64, 8), (76, 31840, 864, 128, 1), (67, 16256, 5312, 128, 2), (66, 8160, 9568, 128, 4),
       (137, 31552, 736, 192, 1), (129, 13472, 5248, 192, 2), (142, 7872, 8416, 192, 4), (446, 6272, 15136, 256, 2)]


@pytest.mark.parametrize("M,I,H,tokens,splits,act", [(*s, a) for i, s in enumerate(GLU)
                                                     for a in (("gelu", "silu") if i < 3 else ("gelu",))])
def test_prefill_glu_bits(orc, dev, M, I, H, tokens, splits, act):
    """The epilogue's GLU gives alv_glu's bits (pinned to the reference by
    test_glu_bit_exact) for M x I pairs: gate and up rows that pick one
    activation each. Values over the float32 path's range, its edges and the
    queue's: |g| from subnormal to 60, zeros on either side and whole rows of
    them, and a token of equal pairs next to a rounding midpoint in every column."""
    import alveare_amd as aa

    _say(f"GLU bits M={M} I={I} H={H} {act}")
    assert _plan(M, I, H, ffn=1) == (tokens, splits)
    half = H // 2
    rows = np.arange(I)
    ffn = aa.pack_ffn_fused_weights(_picker(I, H, rows % half), _picker(I, H, half + rows // half),
                                    orc.synth_q4(H, I, 5), H, I, activation=act, device=dev)
    g = torch.Generator().manual_seed(M + I)
    x = torch.randn(M, H, generator=g) * torch.exp2(torch.randint(-12, 6, (M, H), generator=g).float())
    x[0] = 0.0
    x[1, :half] = torch.linspace(-12.0, 12.0, half)
    x[2, :half] = -torch.exp2(torch.linspace(-130.0, 5.9, half))
    x[3] = 1.0  # one pair in every column
    x[4, half:] = 0.0  # zero up beside any gate, zero gate beside any up
    x[5, :half] = 0.0
    x[6, :half] = -torch.exp2(torch.linspace(3.0, 127.0, half))  # gates past the exponential's range
    x[6, half:] = 0.0
    x[7, :half] = -torch.linspace(4.0, 40.0, half)  # 1 + tanh from ordinary to zero in float64
    x[M // 2:M // 2 + 8] = 0.0  # rows of zeros inside a tile
    x = x.to(torch.bfloat16).to(dev)
    y = torch.empty(M, H, dtype=torch.bfloat16, device=dev)
    from alveare_amd import layer
    layer.ffn_fused_bf16(ffn, x, y, M)
    got = ffn.last_activation(M)
    cols = torch.from_numpy(rows).to(dev)
    gg = x.float()[:, cols % half].contiguous()
    uu = x.float()[:, half + cols // half].contiguous()
    want = torch.empty_like(gg)
    aa._lib.check(aa.lib().alv_glu(gg.data_ptr(), uu.data_ptr(), want.data_ptr(), gg.numel(),
                                   0 if act == "gelu" else 1, torch.cuda.current_stream().cuda_stream), "alv_glu")
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    # and the down product of that activation
    w64 = aa.dequant_q4(torch.from_numpy(orc.synth_q4(H, I, 5)).to(dev), H, I).double()
    ref = got.double() @ w64.T
    bound = (I + 8) * 2.0 ** -24 * (got.double().abs() @ w64.abs().T) + ref.abs() * 2.0 ** -8 + 1e-30
    assert ((y.double() - ref).abs() <= 1.01 * bound).all()
    ffn.close()


@pytest.mark.parametrize("M,I,H,tokens,splits", [GLU[0], GLU[1], GLU[5], GLU[9], GLU[12]])
@pytest.mark.parametrize("share", [0.01, 0.05, 0.3, 1.0])
def test_prefill_glu_queue(orc, dev, M, I, H, tokens, splits, share):
    """Gates between -7.6 and -5.7, which only the float64 path settles, in a
    hundredth to all of the values: the queue is drained between batches, at its
    limit, and at the tile's end, with the bits of alv_glu."""
    import alveare_amd as aa
    from alveare_amd import layer

    _say(f"GLU queue M={M} I={I} H={H}, {share} of the gates")
    assert _plan(M, I, H, ffn=1) == (tokens, splits)
    half, rows = H // 2, np.arange(I)
    ffn = aa.pack_ffn_fused_weights(_picker(I, H, rows % half), _picker(I, H, half + rows // half),
                                    orc.synth_q4(H, I, 5), H, I, device=dev)
    g = torch.Generator().manual_seed(M + I)
    x = torch.randn(M, H, generator=g)
    band = -5.7 - 1.9 * torch.rand(M, half, generator=g)
    x[:, :half] = torch.where(torch.rand(M, half, generator=g) < share, band, x[:, :half])
    x = x.to(torch.bfloat16).to(dev)
    layer.ffn_fused_bf16(ffn, x, M=M)
    got = ffn.last_activation(M)
    cols = torch.from_numpy(rows).to(dev)
    gg, uu = x.float()[:, cols % half].contiguous(), x.float()[:, half + cols // half].contiguous()
    want = torch.empty_like(gg)
    aa._lib.check(aa.lib().alv_glu(gg.data_ptr(), uu.data_ptr(), want.data_ptr(), gg.numel(), 0,
                                   torch.cuda.current_stream().cuda_stream), "alv_glu")
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    ffn.close()


def test_prefill_scratch_holds_no_old_values(orc, dev):
    """A call whose packed activation is padded (35 blocks of 32: a last
    substep of three) right after one that filled the stream's scratch with NaN."""
    import alveare_amd as aa
    from alveare_amd import layer

    _say("padding after a NaN call")
    big = aa.pack_ffn_fused_weights(orc.synth_q4(2048, 512, 1), orc.synth_q4(2048, 512, 2), orc.synth_q4(512, 2048, 3),
                                    512, 2048, device=dev)
    layer.ffn_fused_bf16(big, torch.full((200, 512), float("nan"), dtype=torch.bfloat16, device=dev), M=200)
    H, I, M = 672, 1120, 45
    Wg, Wu, Wd = orc.synth_q4(I, H, 4), orc.synth_q4(I, H, 5), orc.synth_q4(H, I, 6)
    ffn = aa.pack_ffn_fused_weights(Wg, Wu, Wd, H, I, device=dev)
    x = torch.from_numpy(orc.synth_normal(M * H, 7)).to(dev).view(M, H).to(torch.bfloat16)
    y = layer.ffn_fused_bf16(ffn, x, M=M).view(M, H)
    a = ffn.last_activation(M)
    assert torch.isfinite(a).all()
    ref = a.double() @ aa.dequant_q4(torch.from_numpy(Wd).to(dev), H, I).double().T
    assert (y.double() - ref).abs().max() <= 2.0 ** -8 * ref.abs().max()
    big.close()
    ffn.close()


def test_prefill_ffn_capture_fallback(orc, dev):
    """An FFN captured on a stream whose scratch holds its activation but not its
    packed input runs the LDS tile kernels, the activation row-major: alv_glu's
    bits, and the down product's bound, at every replay."""
    import alveare_amd as aa
    from alveare_amd import layer

    _say("FFN capture without packing scratch")
    H, I, M = 4096, 512, 200  # 1.6 MB packed, 0.2 MB of activation; scratch grows by whole MiB
    half, rows = H // 2, np.arange(I)
    Wd = orc.synth_q4(H, I, 5)
    ffn = aa.pack_ffn_fused_weights(_picker(I, H, rows % half), _picker(I, H, half + rows), Wd, H, I, device=dev)
    small = aa.pack_ffn_fused_weights(orc.synth_q4(512, 64, 1), orc.synth_q4(512, 64, 2), orc.synth_q4(64, 512, 3), 64,
                                      512, device=dev)
    x = torch.from_numpy(orc.synth_normal(M * H, 7)).to(dev).view(M, H).to(torch.bfloat16)
    xs = torch.ones(40, 64, dtype=torch.bfloat16, device=dev)
    w64 = aa.dequant_q4(torch.from_numpy(Wd).to(dev), H, I).double()
    gg, uu = (x[:, c].float().contiguous() for c in (torch.from_numpy(rows % half).to(dev), torch.from_numpy(half + rows).to(dev)))
    want = torch.empty_like(gg)
    y = torch.empty(M * H, dtype=torch.bfloat16, device=dev)
    torch.cuda.synchronize()
    s = torch.cuda.Stream(device=dev)
    with torch.cuda.stream(s):
        aa._lib.check(aa.lib().alv_glu(gg.data_ptr(), uu.data_ptr(), want.data_ptr(), gg.numel(), 0, s.cuda_stream), "alv_glu")
        layer.ffn_fused_bf16(small, xs, M=40)
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            layer.ffn_fused_bf16(ffn, x, y, M)
        ref = want.double() @ w64.T
        bound = (I + 8) * 2.0 ** -24 * (want.double().abs() @ w64.abs().T) * 1.01 + ref.abs() * 2.0 ** -8 + 1e-30
        for _ in range(3):
            y.zero_()
            graph.replay()
            got = ffn.last_activation(M)
            s.synchronize()
            assert torch.equal(got.view(torch.int32), want.view(torch.int32))
            assert ((y.view(M, H).double() - ref).abs() <= bound).all()
            layer.ffn_fused_bf16(small, xs, M=40)
            s.synchronize()
    ffn.close()
    small.close()


def test_prefill_capture(orc, dev):
    """Captured after an eager call of its shape, the packed path replays its
    bits, eager work of other shapes between the replays; captured on a stream
    whose scratch was never sized, the call still runs (the kernel that needs
    no scratch) and agrees within bf16 rounding of the same sums."""
    from alveare_amd import layer

    _say("capture")
    M, N, K = 45, 700, 1056
    w, w64 = _weight(orc, dev, N, K, 11)
    x = torch.from_numpy(orc.synth_normal(M * K, 12)).to(dev).view(M, K).to(torch.bfloat16)
    other = torch.from_numpy(orc.synth_normal(300 * K, 13)).to(dev).view(300, K).to(torch.bfloat16)
    want = layer.gemv_bf16(w, x, M=M).clone()
    ref = x.double() @ w64.T
    bound = (K + 8) * 2.0 ** -24 * (x.double().abs() @ w64.abs().T) * 1.01 + ref.abs() * 2.0 ** -8
    for sized in (True, False):
        s = torch.cuda.Stream(device=dev)
        y = torch.empty(M * N, dtype=torch.bfloat16, device=dev)
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            if sized:
                layer.gemv_bf16(w, x, y, M)
            s.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=s):
                layer.gemv_bf16(w, x, y, M)
            for _ in range(3):
                y.zero_()
                graph.replay()
                s.synchronize()
                if sized:
                    assert torch.equal(y, want)
                assert ((y.view(M, N).double() - ref).abs() <= bound).all()
                if sized:
                    layer.gemv_bf16(w, other, M=300)
                s.synchronize()
    w.close()
