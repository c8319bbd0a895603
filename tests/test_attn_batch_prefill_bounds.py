"""Index bounds of the batched decode attention and the prefill attention tile kernels, modelled on
the CPU (no GPU), as tests/test_attn_bounds.py does for the single-sequence decode kernels.

Every global and LDS index is enumerated over the whole grid and every thread, for the model shapes
the batched paths take (head_dim <= 128, a multiple of 4), several sequence counts and mixed
positions, and checked against its buffer's extent:
  * qmh_launch_bt_attention  quillm_amd/csrc/qmh_batch.hip:222-248: the kernel choice by B, shape
                             and the largest position
  * k_attn_scores<HD> and k_attn_pv_mha<640> over blockIdx.z (qmh_launch_attn_batch,
                             quillm_amd/csrc/qmh_attn.hip:930-950): sequence z at q + z*n_heads*hd,
                             caches at + z*kv_stride, scores at + z*n_heads*max_seq, position pos[z]
  * k_bt_scores / k_bt_softmax / k_bt_pv  quillm_amd/csrc/qmh_batch.hip:16-117
  * k_bt_attn                quillm_amd/csrc/qmh_batch.hip:129-219 (V chunks of 128 positions
                             clamped to position n-1, the scores and probabilities in LDS after the
                             staged V, LDS of BT_FC*128 + max_pos + 1 floats)
  * qmh_launch_pf_attention  quillm_amd/csrc/qmh_prefill.hip, with k_pf_scores_m<HD> (16 x 64 tiles, queries
                             in LDS below 128 dimensions, positions clamped to max_seq - 1),
                             k_pf_softmax_r<R, W> (W waves per row, the exponentials in LDS for W > 1) and
                             k_pf_pv_m<HD> (sets of 8 positions loaded two ahead, the reversed second half
                             of the token groups and Wo's quantized image). A buffer load that runs past
                             what is used is in bounds when its resource lies in the array and nothing but
                             the lane's offset, which the range check covers, is added to its base
The batched caches are [n_layers][B][kvd * max_seq] (qmh_batch_create, kv_stride = kvd*max_seq,
quillm_amd/host/qmh_host.c:1337): a sequence's index past its own stride would read the next
sequence's cache (or, for the last one, past the allocation), so the checks hold each sequence
to its own stride. This is a model: a kernel edit that changes an index must change it here too.
"""
import numpy as np
import pytest

from test_attn_bounds import CW, LDS_MAX, SC_T, WG, Extents, inb, pv, scores

BT_T, BT_FC, BT_FUSE_MAX, BT_DECODE_B, BT_VC = 1024, 128, 16384, 3, 64
PF_VC, PF_TOK = 64, 16

# (n_heads, n_kv_heads, head_dim, max_seq): the batched paths' shapes (head_dim <= 128, multiple of 4)
SHAPES = [
    (6, 6, 48, 256), (6, 2, 48, 256), (12, 12, 64, 1024), (32, 4, 64, 2048), (32, 32, 128, 640),
    (4, 2, 16, 64), (3, 3, 32, 48), (12, 1, 8, 300), (4, 2, 48, 136), (2, 2, 128, 1300), (4, 2, 32, 700),
]


def seq_positions(S, B, seed):
    """B positions in [0, S): mixed, with the first at S-1 and the second at 0 when B allows."""
    rng = np.random.default_rng(seed)
    p = rng.integers(0, S, size=B)
    p[0] = S - 1
    if B > 1:
        p[1] = 0
    return p


class BExt:
    """Extents of the batched step's buffers: B sequences of q/out (n_heads*hd), scores
    (n_heads*max_seq) and caches (one stride each)."""

    def __init__(self, nh, nkv, hd, S, B):
        self.stride = nkv * hd * S
        self.K = self.V = B * self.stride
        self.q = self.out = B * nh * hd
        self.att = B * nh * S


def in_seq(what, idx, b, stride):
    """the index of sequence b stays in its own cache region"""
    idx = np.asarray(idx)
    if idx.size:
        assert idx.min() >= b * stride and idx.max() < (b + 1) * stride, f"{what}: sequence {b} leaves its cache"


def attn_batch(nh, nkv, hd, S, pos, e):
    """qmh_launch_attn_batch: the single-sequence kernels with blockIdx.z = sequence. Each sequence's
    indices are the single-sequence kernels' (checked by their own models against one sequence's
    extents) plus the sequence's base offsets, which must keep it inside its own region."""
    one = Extents(nh, nkv, hd, S)
    assert one.K == e.stride and one.V == e.stride  # kv_stride = kvd * max_seq holds one sequence
    for z, p in enumerate(pos):
        scores(nh, nkv, hd, S, int(p), one)
        pv(nh, nkv, hd, S, int(p), one)
        # the z bases of the two kernels (k_attn_scores: q, Kt, att; k_attn_pv_mha: att, V, out)
        inb("batch q base", z * nh * hd + one.q - 1, e.q)
        inb("batch att base", z * nh * S + one.att - 1, e.att)
        inb("batch out base", z * nh * hd + one.out - 1, e.out)
        in_seq("batch K base", z * e.stride + np.array([0, one.K - 1]), z, e.stride)


def bt_scores(nh, nkv, hd, S, pos, e):
    """k_bt_scores over grid (n_heads, B, max_pos/256 + 1) x 256 threads."""
    group, D = nh // nkv, nh * hd
    nz = int(pos.max()) // WG + 1
    tid = np.arange(WG)
    assert hd <= 256  # qs[256]
    for b, p in enumerate(pos):
        for z in range(nz):
            if z * WG > p:
                continue
            t = z * WG + tid
            for h in range(nh):
                inb("bt q", b * D + h * hd + tid[tid < hd], e.q)
                tt = t[t <= p]
                kvh = h // group
                d = np.minimum(np.arange(((hd + 63) // 64) * 64), hd - 1)
                k = b * e.stride + kvh * hd * S + tt[None, :] + d[:, None] * S
                inb("bt K", k, e.K)
                in_seq("bt K", k, b, e.stride)
                inb("bt att", (b * nh + h) * S + tt, e.att)


def bt_softmax(nh, S, pos, e):
    """k_bt_softmax over grid (n_heads, B) x 256 threads: the row of (sequence, head) in place."""
    for b, p in enumerate(pos):
        n = int(p) + 1
        for h in range(nh):
            inb("bt softmax row", (b * nh + h) * S + np.arange(n), e.att)


def bt_pv(nh, nkv, hd, S, pos, e):
    """k_bt_pv over grid (n_heads, B) x 256 threads: V through LDS 64 positions at a time."""
    group, kvd, hd4 = nh // nkv, nkv * hd, hd // 4
    VR = BT_VC * 32 // WG
    tid = np.arange(WG)
    ek = (np.arange(VR)[:, None] * WG + tid[None, :]).ravel()
    t_l, c4 = ek >> 5, ek & 31
    inb("bt pv LDS vs", t_l * 128 + 4 * c4 + 3, BT_VC * 128)
    for b, p in enumerate(pos):
        n = int(p) + 1
        for h in range(nh):
            kvh = h // group
            for c0 in range(0, n, BT_VC):
                tc = np.minimum(c0 + t_l, n - 1)
                on = c4 < hd4
                v = b * e.stride + kvh * hd + tc[on] * kvd + 4 * c4[on] + 3
                inb("bt pv V", v, e.V)
                in_seq("bt pv V", v, b, e.stride)
                pr = c0 + tid[tid < BT_VC]
                inb("bt pv P", (b * nh + h) * S + pr[pr < n], e.att)
            inb("bt pv out", b * nh * hd + h * hd + tid[tid < hd], e.out)


def bt_attn(nh, nkv, hd, S, pos, e):
    """k_bt_attn over grid (n_heads, B) x 1024 threads, LDS BT_FC*128 + max_pos + 1 floats."""
    group, kvd, hd4 = nh // nkv, nkv * hd, hd // 4
    max_pos = int(pos.max())
    lds = BT_FC * 128 + max_pos + 1
    assert 4 * lds <= LDS_MAX
    VR = BT_FC * 32 // BT_T
    tid = np.arange(BT_T)
    ek = (np.arange(VR)[:, None] * BT_T + tid[None, :]).ravel()
    t_l, c4 = ek >> 5, ek & 31
    inb("bt attn LDS vs", t_l * 128 + 4 * c4 + 3, BT_FC * 128)
    for b, p in enumerate(pos):
        n = int(p) + 1
        assert n <= max_pos + 1
        inb("bt attn LDS P", BT_FC * 128 + np.arange(n), lds)
        for h in range(nh):
            kvh = h // group
            inb("bt attn q", b * nh * hd + h * hd + tid[tid < hd], e.q)
            for c0 in range(0, n, BT_FC):
                tc = np.minimum(c0 + t_l, n - 1)
                on = c4 < hd4
                v = b * e.stride + kvh * hd + tc[on] * kvd + 4 * c4[on] + 3
                inb("bt attn V", v, e.V)
                in_seq("bt attn V", v, b, e.stride)
                inb("bt attn P read", BT_FC * 128 + np.minimum(c0 + t_l, n - 1), lds)
            for t0 in range(0, n, BT_T):
                t = t0 + tid[(t0 + (tid & ~63)) < n]  # whole waves past n leave
                tc = np.minimum(t, n - 1)
                d = np.minimum(np.arange(((hd + 31) // 32) * 32), hd - 1)
                k = b * e.stride + kvh * hd * S + d[:, None] * S + tc[None, :]
                inb("bt attn K", k, e.K)
                in_seq("bt attn K", k, b, e.stride)
            inb("bt attn out", b * nh * hd + h * hd + tid[tid < hd], e.out)


def bt_attention(nh, nkv, hd, S, pos, split=0):
    """qmh_launch_bt_attention's choice for B sequences at positions pos."""
    B = len(pos)
    e = BExt(nh, nkv, hd, S, B)
    assert 4 <= hd <= 128 and hd % 4 == 0 and nh % nkv == 0 and 0 <= pos.max() < S
    if split == 0 and B <= BT_DECODE_B and nh == nkv and hd in (128, 64, 48):
        attn_batch(nh, nkv, hd, S, pos, e)
        return "single-sequence kernels"
    if split != 1 and pos.max() < BT_FUSE_MAX:
        bt_attn(nh, nkv, hd, S, pos, e)
        return "k_bt_attn"
    bt_scores(nh, nkv, hd, S, pos, e)
    bt_softmax(nh, S, pos, e)
    bt_pv(nh, nkv, hd, S, pos, e)
    return "three kernels"


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("B", [1, 2, 3, 4, 16])
def test_batched_decode_attention_indices_in_bounds(shape, B):
    nh, nkv, hd, S = shape
    for seed in range(2):
        pos = seq_positions(S, B, seed)
        bt_attention(nh, nkv, hd, S, pos)
        # the split paths too (split 1: three kernels; 2: the fused kernel past BT_DECODE_B's rule)
        bt_attention(nh, nkv, hd, S, pos, split=1)
        bt_attention(nh, nkv, hd, S, pos, split=2)


def test_batched_decode_kernel_choice():
    pos = np.array([5, 9, 100])
    assert bt_attention(32, 32, 128, 640, pos) == "single-sequence kernels"
    assert bt_attention(32, 4, 64, 2048, pos) == "k_bt_attn"  # grouped heads: not the z grid
    assert bt_attention(32, 32, 128, 640, np.arange(4)) == "k_bt_attn"  # past BT_DECODE_B sequences
    assert bt_attention(32, 32, 128, 640, pos, split=1) == "three kernels"


def test_batched_model_catches_a_sequence_leaving_its_cache():
    """Not vacuous: a V row index formed with the query head's index instead of its kv head's, in
    the three-kernel path of grouped heads, leaves the sequence's cache for the last heads."""
    nh, nkv, hd, S, B = 8, 2, 64, 256, 3
    e = BExt(nh, nkv, hd, S, B)
    b, h, tc = B - 1, nh - 1, S - 1
    kvd = nkv * hd
    with pytest.raises(AssertionError):
        in_seq("planted", b * e.stride + h * hd + tc * kvd + np.arange(hd), b, e.stride)


# ---------------------------------------------------------------------------- prefill tiles

def pf_scores_m(HD, nh, nkv, S, P, pos0, e):
    """k_pf_scores_m<HD> over grid (n_heads, ceil(P/64), ceil((pos0+P)/64)) x 4 waves."""
    group, DG = nh // nkv, 8
    l = np.arange(64)
    if HD < 128:  # the wave's 16 queries as whole rows in LDS, HD + 4 floats apart
        i = (np.arange(HD // 16)[:, None] * 64 + l[None, :]).ravel()
        r, d = i // (HD // 4), 4 * (i % (HD // 4))
        assert np.array_equal(np.sort(r * HD + d), np.arange(0, 16 * HD, 4)), "every float4 of 16 queries once"
        inb("pf scores LDS", r * (HD + 4) + d + 3, 16 * (HD + 4))
    else:
        r, d = l & 15, HD - 4
    d0 = np.arange(0, HD, 2 * DG)  # sets of DG dimensions; the one after the last reads the first again
    dn = np.concatenate([d0 + DG, np.where(d0 + 2 * DG < HD, d0 + 2 * DG, 0)])
    assert dn.max() + DG <= HD
    for p0 in range(0, P, 16):
        for c0 in range(0, pos0 + P, 64):
            if c0 > pos0 + min(p0 + 15, P - 1):
                continue
            tc = np.minimum(c0 + l, S - 1)
            for h in range(nh):
                inb("pf Q", (np.minimum(p0 + r, P - 1) * nh + h) * HD + d + 3, P * nh * HD)
                for dd in (0, HD - 1):
                    inb("pf K", ((h // group) * HD + dd) * S + tc, e.K)
                for el in range(4):
                    pt = p0 + 4 * (l >> 4) + el
                    for b in range(4):
                        t = c0 + 16 * b + (l & 15)
                        on = (pt < P) & (t <= pos0 + pt)
                        inb("pf att", ((h * P + pt) * S + t)[on], nh * P * S)


def pf_softmax(nh, S, P, pos0):
    """k_pf_softmax_r<R, W> (rows up to 64*W*R) or k_pf_softmax: row (head, token) of n = pos0+p+1."""
    rlen = pos0 + P
    R, W = next(((R, W) for R, W in ((2, 1), (4, 1), (8, 1), (4, 4), (8, 4), (16, 4)) if rlen <= 64 * R * W), (0, 0))
    for p in range(P):
        n = pos0 + p + 1
        assert n <= S
        if R:
            assert n <= 64 * W * R  # the buffer range check zeroes the rest; stores are masked by n
        if W > 1:  # the serial sum reads the exponentials in pieces of 64
            inb("pf softmax ex LDS", np.arange(0, n, 64) + 63, 64 * W * R)
        for h in range(nh):
            inb("pf softmax row", (h * P + p) * S + np.arange(n), nh * P * S)


def pf_pv_m(HD, nh, nkv, S, P, pos0, e, PP, in_lane=True):
    """k_pf_pv_m<HD> over grid (n_heads * CG/CW, ceil(P / (16*TW))) x 4 waves, with Wo's image. in_lane: the
    position is in the lane's offset; else in the scalar offset, which must lie in the arrays by itself."""
    NB = 3
    CG = (HD + 31) // 32
    CW = 4 if CG % 4 == 0 else 2 if CG % 2 == 0 else 1
    TW = 4 // CW
    group, kvd = nh // nkv, nkv * HD
    G = (P + 16 * TW - 1) // (16 * TW)
    half, y = (G + 1) // 2, np.arange(G)
    grp = np.where(y < half, G - 1 - y, y - half)
    assert np.array_equal(np.sort(grp), np.arange(G)), "every token group once"
    l = np.arange(64)
    hi, row0 = l >> 5, 4 * (l >> 4)
    nblk = nh * HD // 32
    inb("pf pv tile LDS", (row0 + 3) * 36 + 16 + (l & 15), 16 * 36)
    for p0 in range(0, P, 16):
        np_ = min(16, P - p0)
        tmax = pos0 + p0 + np_
        # sets loaded: two before the loop, then one per set used, two ahead
        sets = sorted({8 * w for w in range(NB - 1)} | {t + 8 * (NB - 1) for t in range(0, tmax, 8)})
        assert sets[-1] + 8 > tmax
        for h in range(nh):
            kvh = h // group
            pbase, vbase = (h * P + p0) * S, kvh * HD
            pl = np.where(p0 + (l & 15) < P, l & 15, np_ - 1)
            for c0 in range(0, 32 * CG, 32):
                cl = np.where(c0 + (l & 31) < HD, c0 + (l & 31), 0)
                for t in sets:
                    po = pl * S + 4 * hi + t
                    vo = cl + (4 * hi + t) * kvd
                    rows = np.maximum(S - np.arange(4), 0)  # V from row j on
                    vn = np.where(rows > 0, rows * kvd - kvh * HD, 0)
                    if not in_lane:
                        inb("pf pv att", pbase + po, nh * P * S)
                        inb("pf pv V", vbase + vo + np.arange(4)[:, None] * kvd, e.V)
                        continue
                    assert 4 * (int(po.max()) + 3) < 1 << 32 and 4 * int(vo.max()) < 1 << 32
                    # the resources lie in their arrays
                    inb("pf pv att resource", np.array([pbase, pbase + np_ * S - 1]), nh * P * S)
                    on = rows > 0
                    inb("pf pv V resource", (vbase + np.arange(4) * kvd + vn - 1)[on], e.V)
                    # and hold every value that is used: positions some token of the group sees
                    for q in range(8):
                        if t + q < tmax:
                            on = hi == q // 4
                            inb("pf pv p used", (po + q % 4)[on], np_ * S)
                            inb("pf pv v used", vo[on], vn[q % 4])
                if c0 + 32 <= HD:
                    kk = np.concatenate([8 * r + (l >> 3) for r in range(2)])
                    on, b = kk < np_, h * (HD // 32) + c0 // 32
                    assert b < nblk
                    inb("pf pv image", ((b * PP + p0 + kk) * 32 + 4 * (np.tile(l, 2) & 7) + 3)[on], nblk * PP * 32)
                    inb("pf pv image d", (b * PP + p0 + kk)[on], nblk * PP)
                for b in range(2):
                    c = c0 + 16 * b + (l & 15)
                    for el in range(4):
                        on = (row0 + el < np_) & (c < HD)
                        inb("pf pv out", (((p0 + row0 + el) * nh + h) * HD + c)[on], P * nh * HD)


# (300, 0), (299, 1), (1, 299), (130, 510) and (9, 1015) end at max_seq of some shape
@pytest.mark.parametrize("HD,nh,nkv,S", [(128, 4, 4, 640), (128, 2, 2, 1300), (64, 3, 3, 1024), (64, 8, 2, 2048),
                                         (64, 4, 1, 300), (48, 6, 2, 300), (48, 2, 1, 4099)])
@pytest.mark.parametrize("P,pos0", [(1, 0), (5, 0), (64, 0), (65, 3), (130, 200), (300, 0), (299, 1), (1, 299),
                                    (130, 510), (9, 1015), (512, 0), (300, 700), (3, 4096)])
def test_prefill_tile_kernel_indices_in_bounds(HD, nh, nkv, S, P, pos0):
    if pos0 + P > S:
        pytest.skip("the launcher takes pos0 + P <= max_seq only")
    e = Extents(nh, nkv, HD, S)
    PP = (min(S, 512) + 127) // 128 * 128  # the model's pf_pp
    if P > PP:
        pytest.skip("a pass holds at most pf_cap tokens")
    pf_scores_m(HD, nh, nkv, S, P, pos0, e)
    pf_softmax(nh, S, P, pos0)
    pf_pv_m(HD, nh, nkv, S, P, pos0, e, PP)


def test_prefill_model_catches_an_unclamped_position():
    """Not vacuous: k_pf_scores_m reads positions c0 .. c0+63 clamped to max_seq-1; without the clamp the last
    tile of a context ending at max_seq = 1300 reads past the last kv head's K."""
    HD, nkv, S = 128, 2, 1300
    K = Extents(2, nkv, HD, S).K
    c0 = 1280
    t = c0 + np.arange(64)
    inb("kept clamp", ((nkv - 1) * HD + HD - 1) * S + np.minimum(t, S - 1), K)
    with pytest.raises(AssertionError):
        inb("planted", ((nkv - 1) * HD + HD - 1) * S + t, K)


@pytest.mark.parametrize("P,pos0", [(1, 0), (1, 299), (300, 0)])
def test_prefill_model_catches_positions_in_the_scalar_offset(P, pos0):
    """Not vacuous: with the position in the scalar offset, which the range check need not cover, the sets
    that P.V loads ahead leave V at the end of a context, and the probabilities of a single token."""
    e = Extents(4, 1, 64, 300)
    with pytest.raises(AssertionError):
        pf_pv_m(64, 4, 1, 300 if pos0 + P > 1 else 8, P, pos0, e, 128 if P == 1 else 512, in_lane=False)
