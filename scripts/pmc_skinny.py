#!/usr/bin/env python3
"""Run only the split decode product on the down-projection shape (64 x 18944
by 3584 x 18944), for rocprofv3 --pmc counter collection."""

import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import torch

import arks_amd.ops as O


def main():
    torch.manual_seed(0)
    M, N, K = 64, 3584, 18944
    a = torch.randn(M, K, dtype=torch.bfloat16, device="cuda")
    w = torch.randn(N, K, dtype=torch.bfloat16, device="cuda") * 0.05
    for _ in range(50):
        O.skinny_gemm(a, w)
    torch.cuda.synchronize()


if __name__ == "__main__":
    main()
