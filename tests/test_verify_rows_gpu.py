"""The row-major verify at the edges of its K quarters and vocabulary tiles: fewer K steps than quarters,
cuts inside a two-step stage, K off the 32-wide step, one vocabulary row, a tile's edge and past it, more
tiles than workgroups fit at once. Decisions and the proposals' own logits bit for bit on the four-quarter
logits of the packed GEMM (test_verify_gpu.run_case)."""

from __future__ import annotations

import pytest
import torch

import oracle
from plm_amd.fast_gemm import hip_linear_f32
from plm_amd.verify import LOGITS_CONFIG, ROWMAJOR_LOGITS_CONFIG, lm_head_verify
from test_verify_gpu import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,V,K", [(1, 1, 8), (5, 127, 40), (16, 128, 96), (17, 129, 232), (33, 1000, 1064),
                                   (48, 4097, 1416), (64, 3000, 2056), (56, 140000, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_quarters_and_tiles(device, R, V, K, dtype):
    print(f"row-major verify R={R} V={V} K={K} {dtype}", flush=True)
    g = torch.Generator(device=device).manual_seed(R + V + K)
    x = torch.randn(R, K, generator=g, device=device).to(dtype)
    w = (torch.randn(V, K + 8, generator=g, device=device) / K ** 0.5).to(dtype)[:, :K]   # rows K + 8 apart
    pending = torch.randint(-1, V + 1, (R,), generator=g, device=device, dtype=torch.int64)
    mode = "bf16" if dtype == torch.bfloat16 else "fp16"
    for m in ("fp32", mode):
        for _ in range(2):   # the second launch finds the first one's counters
            run_case(x, w, pending, 0.7, m, device, check_cpu=False, packed=False)


# few_rows_kernel: one row, both pipelines (K steps per wavefront up to four, and more), K off the step and
# fewer steps than quarters, the last row of its range and the next one, more tiles than workgroups.
@pytest.mark.parametrize("R,V,K", [(1, 8192, 512), (2, 33, 8), (4, 1001, 520), (7, 4097, 2056), (8, 4097, 2056),
                                   (14, 300, 4096), (15, 300, 4096), (2, 31000, 4104)])
def test_few_rows(device, R, V, K):
    test_quarters_and_tiles(device, R, V, K, torch.bfloat16)
    test_quarters_and_tiles(device, R, V, K, torch.float16)


@pytest.mark.parametrize("packed", [True, False], ids=["packed", "rowmajor"])
@pytest.mark.parametrize("R,V,K", [(3, 1, 8), (5, 129, 64), (16, 5003, 64), (42, 300, 2048), (64, 20000, 64)])
def test_rows_of_minus_infinity_name_their_first_id(device, R, V, K, packed):
    """Logits that round to -inf in fp16: a row of nothing else has argmax 0, a row with a finite logit
    in a later tile that one's id."""
    x = torch.zeros(R, K, device=device).half()
    w = torch.full((V, K), -300.0, device=device).half()
    w[V // 2, 1] = 1.0
    x[0] = 300.0
    x[1, 0] = 300.0
    x[2, 1] = 300.0
    pending = torch.zeros(R, dtype=torch.int64, device=device)
    argmax = lm_head_verify(x, w, pending, 0.7, "fp16", packed=packed)[1]
    logits = hip_linear_f32(x, w, LOGITS_CONFIG if packed else ROWMAJOR_LOGITS_CONFIG).half()
    assert int(logits[:3].isfinite().sum()) == 1 and bool(logits[2, V // 2].isfinite())
    assert torch.equal(argmax.cpu(), oracle.argmax(logits.float().cpu()))
