"""Index bounds of the tiled prefill matmul's staged loads (k_pf_gemm, quillm_amd/csrc/qmh_prefill.hip) and of the f32
matmul (k_gemm_nt, qmh_ops.hip), modelled on the CPU (no GPU) as tests/test_attn_bounds.py does for the decode
attention kernels.

The blocks pass in stages of four, and stages are loaded ahead of the one multiplied, so the last loads
are of blocks past the row's end. Their addresses are a lane offset plus a block offset that a buffer's range
check need not cover: each must lie in its array by itself. The model enumerates every load of every
thread (weight codes and scales, activation codes and scales), stage by stage as the kernel issues them, and
the LDS pieces that a stage writes. A kernel edit that changes an index must change it here too.
"""
import numpy as np
import pytest

from test_attn_bounds import inb

KB = 4
# (interleaved, row tiles, token tiles, stages ahead beyond two): the instances qmh_launch_pf_gemm starts
INSTANCES = [(True, 2, 1, 1), (True, 2, 2, 1), (False, 2, 1, 1), (False, 2, 2, 1), (False, 4, 2, 0)]


def instance(P, rows, il):
    """qmh_launch_pf_gemm's choice among the tiled instances."""
    if il:
        return INSTANCES[0] if P <= 32 else INSTANCES[1]
    if P <= 32:
        return INSTANCES[2]
    return INSTANCES[3] if (P + 63) // 64 * ((rows + 127) // 128) <= 128 else INSTANCES[4]


def stage_starts(nb, deep):
    """the first blocks of the stages k_pf_gemm loads: those before the loop, then one per stage of the
    loop, which takes an even number of them"""
    nst = (nb + KB - 1) // KB
    ahead = 2 + deep
    return [i * KB for i in range(ahead + 1)] + [(i + ahead + 1) * KB for i in range((nst + 1) // 2 * 2)]


def slot0(row, half, nb, tile_r, il):
    h = tile_r // 2 if il else tile_r
    return row // h * nb * tile_r + row % h + half * h * il


def gemm_loads(rows, nb, tile_r, il, P, PP, cb, last_block_again=True):
    """Every address of k_pf_gemm's staged loads. last_block_again: blocks past the end are the last one."""
    _, RT, TT, deep = instance(P, rows, il)
    WG, NR, NTK = 64 * RT * TT, 32 * RT, 32 * TT
    RS, TS = WG // NR, WG // NTK
    NA, NB, ND = KB // RS, 2 * KB // TS, (KB + TS - 1) // TS
    per = tile_r // 2 if il else tile_r
    ntiles = (rows + per - 1) // per
    rows_alloc, slots = ntiles * per, ntiles * tile_r * nb
    tid = np.arange(WG)
    wave = tid // 64
    row, tok, q0 = tid % NR, tid % NTK, tid // NTK
    j0, qb = wave * 64 // NR, wave * 64 // NTK // 2
    assert np.array_equal(j0, tid // NR) and np.array_equal(qb, q0 // 2)
    piece_a, piece_b = KB * RT * 1024, KB * TT * 1024
    stage = piece_a + piece_b + RT * 32 * 8 + TT * 32 * 8

    def blk(b):
        return np.minimum(b, nb - 1) if last_block_again else b

    # a stage's pieces: each (block, row) and (block, half, token) once, inside the stage's LDS
    a = np.concatenate([(j0 + k * RS) * NR + row for k in range(NA)])
    assert np.array_equal(np.sort(a), np.arange(KB * NR))
    inb("LDS codes", np.concatenate([(j0 + k * RS) * (NR * 32) + NR * 16 + row * 16 + 15 for k in range(NA)]), piece_a)
    b = np.concatenate([(q0 + k * TS) * NTK + tok for k in range(NB)])
    assert np.array_equal(np.sort(b), np.arange(2 * KB * NTK))
    inb("LDS activations", piece_a + b * 16 + 15, piece_a + piece_b)
    on = [(tid >= 0) if TS <= KB else wave * 64 // NTK < KB for k in range(ND)]
    d = np.concatenate([(tok * KB + q0 + k * TS)[on[k]] for k in range(ND)])
    assert np.array_equal(np.sort(d), np.arange(KB * NTK))
    inb("LDS scales", piece_a + piece_b + RT * 32 * 8 + 2 * d + 1, stage)

    starts = stage_starts(nb, deep)
    assert max(starts) >= nb  # the stages do run past the end
    step = NR // 2 if il else NR
    for rg0 in range(0, (rows + step - 1) // step * step, step):
        slot_w = slot0(rg0, 0, nb, tile_r, il)
        rr = rg0 + (row % (NR // 2) if il else row)
        slot = slot0(np.where(rr < rows_alloc, rr, rg0), row // (NR // 2) if il else 0, nb, tile_r, il)
        assert (slot >= slot_w).all()  # offsets from the workgroup's first slot are unsigned
        for b0 in starts:
            for k in range(NA):
                s = slot + blk(b0 + j0 + k * RS) * tile_r
                inb("weight codes", s * cb + cb - 1, slots * cb)
                inb("weight scales", s, slots)
    for t0 in range(0, (P + NTK - 1) // NTK * NTK, NTK):
        for b0 in starts:
            for k in range(NB):
                x = (blk(b0 + qb + k * (TS // 2)) * PP + t0 + tok) * 32 + (q0 & 1) * 16 + 15
                inb("activation codes", x, nb * PP * 32)
            for k in range(ND):
                qs = q0 if NTK < 64 else wave * 64 // NTK
                inb("activation scales", (blk(b0 + qs + k * TS) * PP + t0 + tok)[on[k]], nb * PP)


# whole and partial stages and an odd number of them (1 to 13 blocks), rows that end inside a tile and a
# workgroup, tokens at the instances' edges; a full image (P == PP)
@pytest.mark.parametrize("nb", [1, 2, 3, 4, 5, 8, 9, 13])
@pytest.mark.parametrize("P,PP", [(8, 128), (32, 128), (33, 128), (65, 128), (128, 128), (512, 512)])
@pytest.mark.parametrize("rows,tile_r,il", [(24, 8, False), (300, 16, False), (517, 16, False), (2500, 16, False),
                                            (200, 32, True), (330, 64, True)])
def test_staged_loads_in_bounds(rows, tile_r, il, P, PP, nb):
    for cb in (16, 32):
        gemm_loads(rows, nb, tile_r, il, P, PP, cb)


@pytest.mark.parametrize("P,il", [(20, False), (64, False), (512, False), (64, True)])
def test_model_catches_blocks_past_the_end(P, il):
    """Not vacuous: without the last block in their place, the stages past the end leave the arrays."""
    with pytest.raises(AssertionError):
        gemm_loads(4096, 9, 64 if il else 16, il, P, 512, 16, last_block_again=False)


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 1, 3), (15, 17, 31), (16, 16, 32), (33, 31, 33), (17, 65, 257), (100, 7, 96)])
def test_f32_matmul_in_bounds(M, N, K):
    """k_gemm_nt over grid (ceil(N/32), ceil(M/32)) x 4 waves: the loads of every chunk of 32 k (whole ones as
    float4s, the last by element), the wave's LDS, the stores; every output once."""
    KS, LD = 32, 36
    l = np.arange(64)
    lr, lk = l >> 3, 4 * (l & 7)
    nc, nf = (K + KS - 1) // KS, K // KS
    seen = np.zeros((M, N), int)
    for wave in range(4):
        for i0 in range(16 * (wave >> 1), M, 32):
            for j0 in range(16 * (wave & 1), N, 32):
                for h in range(2):
                    for rows, r0 in ((M, i0), (N, j0)):
                        row = np.minimum(r0 + lr + 8 * h, rows - 1)
                        for c in range(nc):
                            for k in range(4):
                                at = c * KS + lk + k
                                on = at >= 0 if c < nf else at < K
                                inb("operand", (row * K + at)[on], rows * K)
                    inb("LDS write", (lr + 8 * h) * LD + lk + 3, 16 * LD)
                for g in range(2):
                    inb("LDS read", (l & 15) * LD + 16 * g + 4 * (l >> 4) + 3, 16 * LD)
                for e in range(4):
                    i, j = i0 + 4 * (l >> 4) + e, j0 + (l & 15)
                    on = (i < M) & (j < N)
                    np.add.at(seen, (i[on], j[on]), 1)
    assert (seen == 1).all()
