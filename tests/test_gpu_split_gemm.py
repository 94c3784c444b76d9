"""GPU: the prefill combine of small products (a tile a workgroup, its groups
split over the wavefronts) against the oracle at every count of groups a
wavefront takes, rows and tokens that end inside a tile, the last size of its
rule and the first past it, flagged tokens and every code width."""
import sys

import numpy as np
import pytest
import torch

import oracle as o

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def pair(nh, n, k, bits, seed):
    w = (o.seeded_normals([n * k], seed)[0] * np.float32(0.02)).astype(np.float32)
    packed, norms = o.cq_pack(w, k, bits=bits)
    return nh.QMat.from_cq(packed, norms, n, k, bits), o.OQMat.from_cq(packed, norms, n, k, bits)


@pytest.mark.parametrize("bits", [4, 2])
@pytest.mark.parametrize("k", [100, 128, 768, 1024, 1100, 2048, 2200, 3000, 4096])
def test_groups(nh, k, bits):
    for n, rows in ((17, 2), (70, 21), (48, 16)):
        say(f"{rows} x {k} x {n}, {bits} bits")
        g, w = pair(nh, n, k, bits, seed=k + n)
        x = o.seeded_normals([rows * k], seed=rows)[0]
        got = g.matmul(nh.QAct.new(torch.from_numpy(x).cuda(), rows, k, bits)).cpu().numpy()
        want = np.asarray(w.matmul(o.OQAct.new(x, rows, k, bits))).reshape(got.shape)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_rule_edges_and_flags(nh):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for k, per_cu in ((256, 2), (2176, 1)):  # 2 groups; 17
        n = 16 * cus // 8
        for tiles in (8 * per_cu, 8 * per_cu + 1):  # the rule's last size, then the general kernel's first
            rows = 16 * tiles - 3
            g, w = pair(nh, n, k, 4, seed=tiles)
            x = o.seeded_normals([rows * k], seed=tiles)[0]
            a = nh.QAct.new(torch.from_numpy(x).cuda(), rows, k, 4)
            flags = torch.from_numpy(np.random.default_rng(tiles).integers(0, 2, rows).astype(np.uint8)).cuda()
            got, part = g.matmul(a), g.matmul_flags(a, flags)
            want = np.asarray(w.matmul(o.OQAct.new(x, rows, k, 4))).reshape(rows, n)
            assert np.array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32))
            # a flagged token's row is that of a product where it is a block token
            ones = g.matmul_flags(a, torch.ones_like(flags))
            zeros = g.matmul_flags(a, torch.zeros_like(flags))
            pick = torch.where(flags[:, None] != 0, ones, zeros)
            assert torch.equal(part.view(torch.int32), pick.view(torch.int32))
