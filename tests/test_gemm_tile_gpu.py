"""The many-row dequant-GEMM (32x32 tiles) against the oracle, at the edges of its
tiles: rows around the 32 / 64 / 128-row workgroups, columns off the 256-column
blocks, K off the 256-element stages, with and without a K split."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # (type, N, K, Ms)
    (12, 40, 512, (17, 32, 33, 65, 128, 129, 300)),
    (12, 4096, 4096, (64, 333)),      # K split over the CUs
    (12, 22016, 1024, (48,)),
    (14, 272, 1024, (31, 96, 257)),
    (2, 100, 1376, (17, 64, 130)),    # a partial quad, an odd number of 128-element chunks
    (2, 528, 96, (40, 128)),          # less than one stage
    (8, 300, 1440, (33, 64, 200)),
    (8, 4096, 2048, (129,)),
    (1, 257, 416, (17, 64, 129)),
    (1, 2048, 2048, (500,)),
    (2, 4096, 1536, (2080,)),         # 272 blocks: a whole round, then 16 sliced ones
    (12, 17000, 1024, (513, 640)),    # a last round of 79 blocks
]


@pytest.mark.parametrize("wtype,N,K,Ms", CASES)
def test_tile_gemm_matches_oracle(ctx, ora, rng, wtype, N, K, Ms):
    if wtype in (2, 12):
        W = ora.synth_q4(wtype, 3, N + K, N, K)
    elif wtype == 1:
        W = ora.f2h_fast((rng.standard_normal((N, K)) * 0.05).astype(np.float32)).view(np.uint8).reshape(-1)
    else:  # random bytes with finite block scales
        bs, ts, at = (32, 34, 0) if wtype == 8 else (256, 210, 208)
        W = rng.integers(0, 256, (N * K // bs, ts), dtype=np.uint8)
        d = (rng.standard_normal(N * K // bs) * 0.01).astype(np.float16)
        W[:, at:at + 2] = d.view(np.uint8).reshape(-1, 2)
        W = W.reshape(-1)
    deq = ora.dequantize(wtype, W, N * K).reshape(N, K).astype(np.float64) if wtype != 1 else \
        ora.h2f_fast(W.view(np.uint16)).reshape(N, K).astype(np.float64)
    wid = ctx.weight_upload(wtype, W, N, K)
    for M in Ms:
        print(f"type {wtype} N {N} K {K} M {M}", flush=True)
        X = ora.f2h_fast(rng.standard_normal((M, K)).astype(np.float32))
        xb, yb = ctx.upload(X), ctx.alloc(M * N * 4)
        ctx.copy_in(yb, np.full((M, N), np.nan, np.float32))
        ctx.verify_gemm(wid, xb, M, yb)
        y = ctx.download(yb, np.float32, (M, N))
        x64 = ora.h2f_fast(X).astype(np.float64)
        ref, mag = x64 @ deq.T, np.abs(x64) @ np.abs(deq).T
        # fp32 sums of exact products: K rounding steps of 2^-24 of the partial sums at most (the Q4_K
        # min term is of the size of its products times 4 here); Q6_K weights are rounded to fp16 (2^-11)
        bound = mag * ((K + 16) * 2.0 ** -24 * 4 + (2.0 ** -11 if wtype == 14 else 0.0))
        assert np.all(np.abs(y - ref) <= bound), float((np.abs(y - ref) / mag).max())
        assert np.sqrt(((y - ref) ** 2).sum() / (ref ** 2).sum()) < (4.5e-4 if wtype == 14 else 1.5e-6)
        xb.free()
        yb.free()
