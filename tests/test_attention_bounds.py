"""Host-side range check of the attention kernels' address arithmetic.

Every global and LDS address that att_scores_kernel, att_decode_kernel,
att_wsum_kernel and att_wsum_q4_kernel (mimir-model_amd/csrc/decoder_ops.hip)
and am::scores_kernel, am::wsum_kernel and am::decode_scores_kernel
(attention_mfma.hip) compute is restated here per workgroup of the launch grid
that launch_attention picks, and its extremes are checked against the sizes of
the buffers: the key cache [kv_heads][C][D], the value cache blocked by eight
keys [kv_heads][ceil(C/8)][D][8], q and out [T][H][D], the workspace
[T][H][max_keys], and each kernel's LDS. The visible ranges come from
adversarial end/start indices (negative, past C, past max_keys, empty
ranges), over D = 8..512, one to many queries, slots, max_keys up to the
8192 limit. With the clamps of the restatement taken out the checks fail.
CPU only: nothing here runs a kernel."""
import itertools

import numpy as np
import pytest

LDS_BYTES = 160 * 1024
ATT_DEC_MAXK = 256


def att_range(kend, kstart, t, C, maxk):
    k0 = 0 if kstart is None else min(max(int(kstart[t]), 0), C - 1)
    n = int(kend[t]) + 1 - k0
    n = min(n, C - k0, maxk)
    return k0, max(n, 0)


def clamp(v, hi):
    return min(v, hi)


class Bounds:
    def __init__(self, T, H, Hkv, D, C, maxk, f16):
        self.T, self.H, self.Hkv, self.D, self.C, self.maxk, self.f16 = T, H, Hkv, D, C, maxk, f16
        self.esz = 2 if f16 else 4
        self.kc_len = Hkv * C * D
        self.vc_len = Hkv * ((C + 7) // 8) * 8 * D
        self.ws_len = T * H * maxk

    def vcache_at(self, hk, j, d):
        return ((hk * ((self.C + 7) // 8) + j // 8) * self.D + d) * 8 + j % 8

    def check(self, lo, hi, size, what):
        assert 0 <= lo and hi < size, f"{what}: [{lo}, {hi}] outside [0, {size})"


def check_scores(b, ranges, QT):
    D, C = b.D, b.C
    tiles = (b.maxk + 63) // 64
    for z in range((b.T + QT - 1) // QT):
        r = [ranges[QT * z + i] if QT * z + i < b.T else (0, 0) for i in range(QT)]
        nmax = max(n for _, n in r)
        for h in range(b.H):
            hk = h // (b.H // b.Hkv)
            for tile in range(tiles):
                if tile * 64 >= nmax:
                    continue
                i0 = next(i for i in range(QT) if r[i][1] > 0)
                same = all(n == 0 or k0 == r[i0][0] for k0, n in r)
                loads = [(hk * C + r[i0][0], nmax)] if same else \
                    [(hk * C + k0, n) for k0, n in r if tile * 64 < n]
                for base, nlim in loads:
                    js = (tile * 64, tile * 64 + 63)  # j0 = tile*64 + grp, j1 = j0 + 32
                    a_lo = base + min(js[0], nlim - 1)
                    a_hi = base + min(js[1], nlim - 1)
                    assert a_lo >= hk * C
                    b.check(a_lo * D, a_hi * D + D - 1, b.kc_len, "scores: key element")
                for i, (_, n) in enumerate(r):
                    if tile * 64 < n:
                        t = QT * z + i
                        b.check((t * b.H + h) * D, (t * b.H + h) * D + D - 1, b.T * b.H * D, "scores: q")
                        jw = min(tile * 64 + 63, n - 1)
                        assert jw < b.maxk
                        b.check((t * b.H + h) * b.maxk, (t * b.H + h) * b.maxk + jw, b.ws_len, "scores: out")


def check_decode(b, ranges):
    D, C, DG = b.D, b.C, 32
    PPB, VPAD = (1, 8) if b.f16 else (2, 4)
    mk = (b.maxk + 3) & ~3
    vstride = ((b.maxk + 14) & ~7) + VPAD
    lds = mk * 4 + DG * vstride * b.esz
    assert lds <= LDS_BYTES - 64
    for t, (k0, n) in enumerate(ranges):
        if n <= 0:
            continue
        for h in range(b.H):
            hk = h // (b.H // b.Hkv)
            base = hk * C + k0
            # keys j + 64, j + 96 past n: the last key
            b.check(base * D, (base + n - 1) * D + D - 1, b.kc_len, "decode: key element")
            assert n <= mk  # scores sc[j], j < n
            k0a, off = k0 & ~7, k0 - (k0 & ~7)
            nblk = (off + n + 7) >> 3
            for d0 in range(0, D, DG):
                src = b.vcache_at(hk, k0a, d0)
                last = src + ((nblk - 1) * D + DG - 1) * 8 + (PPB - 1) * 4 + 16 // b.esz - 1
                b.check(src, last, b.vc_len, "decode: value element")
                # LDS dim rows: writes up to 8*nblk, chain reads up to off + n
                assert 8 * nblk <= vstride and off + n <= vstride
                assert (DG - 1) * vstride + 8 * nblk <= DG * vstride


def check_wsum(b, ranges):
    D, C = b.D, b.C
    PPB, BB, NR = (1, 16, 4) if b.f16 else (2, 16, 3)
    CPB = BB // 2 if b.f16 else BB  # copies a batch a copying wave (waves 1 and 2)
    batch = BB * PPB * 1024
    e_len = (b.maxk + 14) & ~7
    assert NR * batch + e_len * 4 + 64 <= LDS_BYTES
    assert 16 * 63 + 16 + ((BB - 1) * PPB + PPB - 1) * 1024 <= batch  # a lane's slot reads and copies
    for t, (k0, n) in enumerate(ranges):
        if n <= 0:
            continue
        k0a, off = k0 & ~7, k0 - (k0 & ~7)
        nb = (off + n + 7) >> 3
        nv = n & ~7 if n >= 8 else 0
        assert off + n - 1 < e_len  # e[off + j]; the exps' clamped reads e[off + min(j, nv - 1)], e[off + nv + tid]
        for bt in range((nb + BB - 1) // BB):  # a whole batch's chain reads e[8*b0 .. 8*(b0+BB)) only when inside
            b0 = BB * bt
            if 8 * b0 >= off and 8 * (b0 + BB) <= off + n:
                assert 8 * (b0 + BB) <= e_len
        # copies: NR - 1 batches ahead of batch 0 and one a batch after, blocks past nb: the last again
        assert (NR - 1) * CPB <= 63  # copies in flight a copying wave (vmcnt)
        for h in range(b.H):
            hk = h // (b.H // b.Hkv)
            for d0 in range(0, D, 64):
                for lane in (0, 63):
                    d = min(d0 + lane, D - 1)
                    for w1 in range(PPB):
                        src = b.vcache_at(hk, k0a, d) + 4 * w1
                        last = src + (nb - 1) * 8 * D + 16 // b.esz - 1  # blocks past nb: the last again
                        b.check(src, last, b.vc_len, "wsum: value element")
                # scores: loads of j and, past the end, the last key (j clamped to n - 1)
                b.check((t * b.H + h) * b.maxk, (t * b.H + h) * b.maxk + n - 1, b.ws_len, "wsum: scores")


def check_wsum_q4(b, ranges):
    D, C = b.D, b.C
    VC, VS = (128, 136) if b.f16 else (64, 76)
    PPB = 1 if b.f16 else 2
    mkp = (b.maxk + 3) & ~3
    assert 4 * mkp * 4 + VS * 64 * b.esz <= LDS_BYTES
    for z in range((b.T + 3) // 4):
        r = [ranges[4 * z + i] if 4 * z + i < b.T else (0, 0) for i in range(4)]
        ns = [n for _, n in r]
        nmax = max(ns)
        first = next((i for i in range(4) if ns[i] > 0), -1)
        same = all(n == 0 or k0 == r[first if first >= 0 else 0][0] for k0, n in r)
        for n in ns:
            assert n <= mkp
        for h in range(b.H):
            hk = h // (b.H // b.Hkv)
            for pas in range(1 if same else 4):
                src = (first if first >= 0 else 0) if same else pas
                pn = nmax if same else ns[pas]
                for c0 in range(0, pn, VC):
                    rows = min(pn - c0, VC)
                    ka = r[src][0] + c0
                    kaa, offc = ka & ~7, ka - (ka & ~7)
                    nblk = (offc + rows + 7) >> 3
                    for d0 in range(0, D, 64):
                        s0 = b.vcache_at(hk, kaa, d0)
                        last = s0 + ((nblk - 1) * D + 63) * 8 + (PPB - 1) * 4 + 16 // b.esz - 1
                        b.check(s0, last, b.vc_len, "wsum_q4: value element")
                    assert 8 * nblk <= VS and offc + rows <= VS


def row_of(b, ranges, hk, rho):
    """am::row_of: first key, keys (none past the last row), t * H + h."""
    G = b.H // b.Hkv
    rows = b.T * G
    rc = clamp(rho, rows - 1)
    t = rc // G
    k0, n = ranges[t] if rc == rho else (0, 0)
    return k0, n, t * b.H + hk * G + rc - t * G


def check_scores_mfma(b, ranges):
    """am::scores_kernel: 32 rows a workgroup, 32 keys a wave, tiles of 128
    keys gridDim.y apart from the rows' first key on."""
    D, C, G = b.D, b.C, b.H // b.Hkv
    rows = b.T * G
    xt = (rows + 31) // 32 * b.Hkv
    gy = max(1, min(1024 // xt, ((C if b.kstart else b.maxk) + 127) // 128))
    for hk in {0, b.Hkv - 1}:
        for rho0 in range(0, rows, 32):
            r = [row_of(b, ranges, hk, rho0 + i) for i in range(32)]
            for i, (_, _, head) in enumerate(r):
                if rho0 + i < rows:
                    b.check(head * D, head * D + D - 1, b.T * b.H * D, "scores_mfma: q")
                b.check(i * (D + 4), i * (D + 4) + D - 1, 32 * (D + 4), "scores_mfma: q row in LDS")
            live = [x for x in r if x[1] > 0]
            if not live:
                continue
            kmin, kfin = min(k0 for k0, _, _ in live), max(k0 + n for k0, n, _ in live)
            walked = []
            for y in range(gy):
                for kt in range(kmin + 128 * y, kfin, 128 * gy):
                    walked.append(kt)
                    for w in range(4):
                        kb = kt + 32 * w
                        seen = [x for x in live if x[0] < kb + 32 and x[0] + x[1] > kb]
                        if not seen:
                            continue
                        a_lo, a_hi = clamp(kb, C - 1), clamp(kb + 31, C - 1)
                        b.check((hk * C + a_lo) * D, (hk * C + a_hi) * D + D - 1, (hk + 1) * C * D, "scores_mfma: key")
                        for k0, n, head in seen:
                            j_lo, j_hi = max(kb - k0, 0), min(kb + 31 - k0, n - 1)
                            b.check(head * b.maxk + j_lo, head * b.maxk + j_hi, (head + 1) * b.maxk, "scores_mfma: out")
            assert sorted(walked) == list(range(kmin, kfin, 128))  # every key's tile once
            assert max(x[2] for x in live) < b.T * b.H


def check_wsum_mfma(b, ranges, RT, each):
    """am::wsum_kernel: RT rows and 64 dims a wave, one first key at a time."""
    D, C, G = b.D, b.C, b.H // b.Hkv
    rows, RG = b.T * G, 1 if each else 2
    R, NT = RG * RT, RG * D
    KC = 64 if RT == 16 else D
    ES, HB = KC + 4, 4 if RT == 16 else KC // (16 if b.f16 else 32)
    SEG = KC // 8 // HB
    assert 8 * HB * SEG == KC and SEG % 2 == 0 and R * KC % NT == 0 and NT % KC in (0, NT) and KC % 64 == 0
    assert 2 * R * ES * 4 + R * (8 + 8 + 1 + 1 + 1 + 1 + 1) * 4 <= LDS_BYTES // 2  # two workgroups a CU
    b.check(0, (R - 1) * ES + 8 * HB * (SEG - 1) + 8 * HB - 1, R * ES, "wsum_mfma: weights read by the chains")
    b.check(0, (R - 1) * ES + 7 + 8 * (KC // 8 - 1), R * ES, "wsum_mfma: weights read by the lane sums")
    for hk in {0, b.Hkv - 1}:
        for rho0 in range(0, rows, R):
            r = [row_of(b, ranges, hk, rho0 + i) for i in range(R)]
            for _, _, head in r:  # every row's scores are loaded, of a row without a key the first word
                b.check(head * b.maxk, head * b.maxk, b.ws_len, "wsum_mfma: a row's first score")
            for i, (_, n, head) in enumerate(r):
                if rho0 + i < rows:
                    b.check(head * D, head * D + D - 1, b.T * b.H * D, "wsum_mfma: out")
                assert n == 0 or rho0 + i < rows
            firsts = list(dict.fromkeys(k0 for k0, n, _ in r if n > 0))
            if each:
                assert len(firsts) <= (G + 2) // G + 1  # a workgroup for each
            for k0 in firsts:
                nall = max(n for k, n, _ in r if n > 0 and k == k0)
                off = k0 & 7
                kbeg, nch, nblk = k0 - off, (off + nall + KC - 1) // KC, (off + nall + 7) >> 3
                for k, n, head in r:
                    un = n if k == k0 else 0
                    # slots -off .. of the first chunk to the last one's end, and the last n % 8 keys
                    for j in (-off, KC * (nch - 1) + KC - 1 - off, (un & ~7) + 7, nall + 63):
                        at = max(clamp(j, un - 1), 0)
                        b.check(head * b.maxk, head * b.maxk + at, (head + 1) * b.maxk, "wsum_mfma: scores")
                last = clamp(HB * (SEG * (nch - 1) + SEG) + HB - 1, nblk - 1)  # one segment read ahead
                for d in (0, D - 1):
                    b.check(b.vcache_at(hk, kbeg, d), b.vcache_at(hk, kbeg + 8 * last, d) + 7, b.vcache_at(hk + 1, 0, 0),
                            "wsum_mfma: value block")
                assert 8 * HB * SEG * nch >= off + nall  # every key's weight is in a chunk


def check_decode_scores(b, ranges):
    """am::decode_scores_kernel: a wave per 64 keys, kv head and query."""
    D, C, G = b.D, b.C, b.H // b.Hkv
    PC, NG = D * b.esz // 16, 1 if G <= 4 else 2
    sw = lambda k: k & (PC - 1) & 15
    for k in range(64):  # the swizzle moves a key's pieces within the key
        assert sorted(p ^ sw(k) for p in range(PC)) == list(range(PC))
    b.check(0, 1024 * (PC - 1) + 16 * 63 + 15, 64 * PC * 16, "decode_scores: pieces in LDS")
    b.check(0, (4 * NG - 1) * (D + 4) + D - 1, 4 * NG * (D + 4), "decode_scores: q rows in LDS")
    for t, (k0, n) in enumerate(ranges):
        for hk in {0, b.Hkv - 1}:
            head0 = t * b.H + hk * G
            for j0 in range(0, min(n, b.maxk), 64):
                lo, hi = clamp(j0, n - 1), clamp(j0 + 63, n - 1)
                b.check((hk * C + k0 + lo) * D, (hk * C + k0 + hi) * D + D - 1, (hk + 1) * C * D, "decode_scores: key")
                heads = [head0 + 4 * g + i for g in range(NG) for i in range(4) if 4 * g + i < G]
                b.check(min(heads) * D, (head0 + clamp(4 * NG - 1, G - 1)) * D + D - 1, b.T * b.H * D, "decode_scores: q")
                j = min(j0 + 63, n - 1)
                b.check(min(heads) * b.maxk + j0, max(heads) * b.maxk + j, (head0 + G) * b.maxk, "decode_scores: out")
            assert n <= b.maxk


def check_scores_gqa(b, ranges):
    """att_scores_gqa_kernel: a workgroup per 64 keys, kv head and query."""
    D, C, G = b.D, b.C, b.H // b.Hkv
    for t, (k0, n) in enumerate(ranges):
        for hk in {0, b.Hkv - 1}:
            head0 = t * b.H + hk * G
            b.check(head0 * D, (head0 + G) * D - 1, b.T * b.H * D, "scores_gqa: q")
            for j0 in range(0, min(n, b.maxk), 64):
                lo, hi = clamp(j0, n - 1), clamp(j0 + 63, n - 1)
                b.check((hk * C + k0 + lo) * D, (hk * C + k0 + hi) * D + D - 1, (hk + 1) * C * D, "scores_gqa: key")
                b.check(head0 * b.maxk + j0, (head0 + G - 1) * b.maxk + min(j0 + 63, n - 1), (head0 + G) * b.maxk,
                        "scores_gqa: out")


def run_launch(T, H, Hkv, D, C, maxk, f16, kend, kstart, aligned=True):
    b = Bounds(T, H, Hkv, D, C, maxk, f16)
    b.kstart = kstart is not None
    ranges = [att_range(kend, kstart, t, C, maxk) for t in range(T)]
    for k0, n in ranges:
        assert 0 <= k0 < C and 0 <= n <= min(C - k0, maxk)
    G, decw = H // Hkv, T * H * D // 32
    if D in (64, 128) and maxk <= ATT_DEC_MAXK and (T < 16 or aligned and (decw <= 512 or decw <= 1024 and maxk <= 64)):
        check_decode(b, ranges)
        return "decode"
    if T >= 16 and D in (64, 128) and aligned:
        check_scores_mfma(b, ranges)
        each = b.kstart and G <= 4 and T * G * maxk <= 4 * C
        RT = 16 if (T * G + 31) // 32 * Hkv >= 256 and not each else 4
        check_wsum_mfma(b, ranges, RT, each)
        return "each" if each else f"mfma{RT}"
    if T >= 16 and D % 64 == 0 and maxk <= 2048:
        check_scores(b, ranges, 4)
        check_wsum_q4(b, ranges)
        return "many"
    kvw = (maxk + 63) // 64 * Hkv * T
    if kvw >= 256 and (G == 2 and (f16 and D == 128 and kvw < 8192 or not f16 and D in (64, 128))
                       or G == 4 and not f16 and D == 128):
        check_scores_gqa(b, ranges)
        check_wsum(b, ranges)
        return "two_gqa"
    if D in (64, 128) and 2 <= G <= 8 and aligned and kvw >= 256:
        check_decode_scores(b, ranges)
        check_wsum(b, ranges)
        return "two_grouped"
    check_scores(b, ranges, 1)
    check_wsum(b, ranges)
    return "two"


def ranges_for(T, C, maxk, slots, rng):
    """End/start indices of T queries in `slots` slots of C entries, with
    adversarial values mixed in: negative, past C, empty, past max_keys."""
    L = C // slots
    kend = np.empty(T, np.int64)
    kstart = np.empty(T, np.int64)
    for t in range(T):
        s = t % slots
        kstart[t] = s * L
        kend[t] = s * L + rng.integers(0, L)
    special = [(-5, -1), (C + 9, C + 3), (C - 1, C - 1), (0, C - 1), (C - 1, 0), (7, 3), (maxk + 50, 0),
               (C * 2, -7), (C - 1, C - 9)]
    for t in range(min(T, len(special))):
        kend[t], kstart[t] = special[t]
    return kend, kstart


@pytest.mark.parametrize("D", [8, 32, 64, 96, 128, 256, 512])
@pytest.mark.parametrize("f16", [True, False])
def test_attention_addresses_in_bounds(D, f16):
    rng = np.random.default_rng(D + (1000 if f16 else 0))
    seen = set()
    for T, (H, Hkv), C, slots, maxk_kind, aligned in itertools.product(
            (1, 3, 8, 16, 37, 300), ((4, 1), (8, 2), (4, 4), (16, 8), (24, 8), (32, 8)), (1, 7, 42, 301, 2048, 8200), (1, 3, 40),
            ("C", "slot", "small", "max"), (True, False)):
        if H in (16, 24) and (T != 8 or C != 2048 or D not in (64, 128)):
            continue
        if slots > C or (H == 32 and T != 300) or (not aligned and (D not in (64, 128) or C > 301)):
            continue
        if (slots == 40) != (maxk_kind == "slot") or (slots == 40 and D not in (64, 128)):
            continue
        maxk = {"C": min(C, 8192), "slot": min(C // slots, 8192), "small": max(1, min(C, 8192) // 3), "max": 8192}[maxk_kind]
        if T * maxk > 8 * 8192 * 37 or (H == 32 and maxk > 2048):
            continue
        kend, kstart = ranges_for(T, C, maxk, slots, rng)
        seen.add(run_launch(T, H, Hkv, D, C, maxk, f16, kend, kstart if slots > 1 or T > 5 else None, aligned))
    if D in (64, 128):
        gqa = set() if f16 and D == 64 else {"two_gqa"}
        assert seen == {"mfma4", "mfma16", "each", "many", "decode", "two", "two_grouped"} | gqa
    elif D % 64 == 0:
        assert seen == {"many", "two"}
    else:
        assert seen == {"two"}


@pytest.mark.parametrize("T,H,Hkv,C,slots,maxk,path", [(37, 4, 4, 301, 1, 301, "mfma4"), (300, 32, 8, 301, 1, 301, "mfma16"),
                                                      (37, 16, 16, 37 * 20, 37, 20, "each"), (8, 8, 2, 2047, 1, 2047, "two_grouped")])
def test_missing_clamps_are_found(monkeypatch, T, H, Hkv, C, slots, maxk, path):
    """The checks of the matrix-core kernels fail when the restatement's
    clamps (rows past the last, keys and value blocks past the end) go."""
    rng = np.random.default_rng(T)
    for t0 in range(3):
        kend, kstart = ranges_for(T, C, maxk, slots, rng)
        kend[-1], kstart[-1] = C - 1, max(0, C - maxk)
        args = (T, H, Hkv, 64, C, maxk, True, kend, kstart if slots > 1 else None)
        assert run_launch(*args) == path
        with monkeypatch.context() as m:
            m.setitem(globals(), "clamp", lambda v, hi: v)
            with pytest.raises((AssertionError, IndexError)):
                run_launch(*args)
