"""Host-side bounds replay of the batch routers: k_route (silentotithrandousha_amd/csrc/
kernels.hip, `k_route<KI, TB, NT, NORM>` and its launcher `launch_route_ki`), and k_route_wide and
k_group (csrc/route_wide.hip): every global and LDS index the kernels compute, enumerated over the whole grid of a launch, against the sizes the library
allocates (moe_api.cpp `carve_work`, `router_bytes`) and the LDS the launch reserves. Covers x
staging (with the norm's passes), the xsplit rows, the router-weight loads, the logit table, the grouped-GEMM activation
records (rec_split_block's byte offsets), the per-wavefront top-k stores, the grouping's
per-block counts and ranks, the last block's count table in the x staging area and its scatter
(a value-dependent index: ge = base[e] + prefix over blocks + rank, replayed on random routings,
so it must land on every entry exactly once), and the per-block timing stamps of the
realtime-counter trace copy (`rt_ts[blockIdx.x * 16 + i]`, i <= 9, over 4096 * 16 entries).

It is a model of the kernels' index arithmetic, not the kernels: it restates each index
expression with a citation of the code it follows, so a change to those expressions needs the
same change here."""
import numpy as np
import pytest

K_ROUTE_THREADS = 1024          # kernels.hip: kRouteThreads
K_ROUTE_TOKENS = 8              # kernels.hip: kRouteTokens
K_MAX_EXPERTS = 256             # kernels.hpp: kMaxExperts
K_MAX_TOPK = 16                 # kernels.hpp: kMaxTopK
K_GEMM_NS = 24                  # kernels.hpp: kGemmNs
K_FINE_TERMS = 6                # kernels.hpp: kFineTerms
LDS_BYTES = 160 * 1024          # gfx950 LDS per workgroup
RT_STAMPS = 4096 * 16           # the trace copy's rt_ts array


def rec_step(nt):               # kernels.hpp GemmRecT<NT>::kStep / kBytes
    return nt * 96 + (4 * nt + 15) // 16 * 16


def row_bytes(nt, H):           # kernels.hpp GemmRecT<NT>::row_bytes: the six-term records hold H's steps only
    return (-(-H // 128) if nt == K_FINE_TERMS else K_GEMM_NS) * rec_step(nt)


def rec_offsets(nt, blk):
    """Byte ranges [lo, hi) rec_split_block writes for block blk (device.hpp rec_split_block,
    GemmRecT::dword / ::scale)."""
    st, i = blk >> 2, blk & 3
    out = []
    for t in range(nt):
        base = st * rec_step(nt) + t * 96
        out.append((base + 16 * i, base + 16 * i + 16))            # dwords 0-3: uint4
        out.append((base + 64 + 8 * i, base + 64 + 8 * i + 8))     # dwords 4-5: uint2
        sc = st * rec_step(nt) + nt * 96 + 4 * t + i
        out.append((sc, sc + 1))                                   # the scale byte
    return out


def launch_shape(T, H):
    """launch_route_ki: TB and the dynamic LDS of the launch."""
    nq = ((H + 63) // 64 + 7) // 8
    hp = nq * 8 * 64                                   # route_hp(H), floats
    if T >= 2048 and K_ROUTE_TOKENS * hp * 4 <= 144 * 1024:
        return nq, hp, K_ROUTE_TOKENS, K_ROUTE_TOKENS * hp * 4
    return nq, hp, 1, hp * 4


def static_lds(TB, norm):
    """k_route's __shared__ arrays in bytes: s_logit, s_p, s_order, s_w, s_sel, s_last, s_cnt, s_r."""
    return 4 * (TB * K_MAX_EXPERTS + K_MAX_EXPERTS + TB * K_MAX_TOPK * 2 + TB + 1 + K_MAX_EXPERTS + (TB if norm else 1))


def check(name, idx, size):
    idx = np.asarray(idx)
    if idx.size:
        lo, hi = int(idx.min()), int(idx.max())
        assert lo >= 0 and hi < size, f"{name}: index range [{lo}, {hi}] outside [0, {size})"


def replay(T, E, k, H, rec_terms=3, xsplit=True, seed=0, stamps=False, norm=False):
    nq, Hp, TB, dyn = launch_shape(T, H)
    KI = nq if nq in (1, 2, 6) else 0
    grid = (T + TB - 1) // TB
    N = T * k
    nw = K_ROUTE_THREADS // 64
    assert dyn + static_lds(TB, norm) <= LDS_BYTES, "LDS of the launch"
    per_wave = k <= 4 and E <= 128
    assert TB < nw                                       # the kernel's static_assert
    lane = np.arange(64)
    rec_bytes = row_bytes(rec_terms, H)
    assert H <= 128 * K_GEMM_NS                           # launch_route: xrec needs H <= 128 kGemmNs
    assert rec_terms != K_FINE_TERMS or (TB == 1 and T * k < 4 * E)  # launch_route_ki, forward_device
    # routing of the replay: k distinct experts per token
    rng = np.random.default_rng(seed)
    order = np.argsort(rng.random((T, E)), axis=1)[:, :k].astype(np.int64)
    blk_count = np.zeros((grid, E), np.int64)
    rank = np.full(N, -1, np.int64)
    for b in range(grid):
        t0 = b * TB
        nt = min(TB, T - t0)
        # x loads and staging (kernels.hip k_route: xv[tb][q], stage(tb, k, xv))
        tb = np.arange(nt)[:, None]
        kk = np.arange(Hp)[None, :]
        check("x", ((t0 + tb) * H + kk)[np.broadcast_to(kk < H, (nt, Hp))], T * H)
        check("s_x staging", (tb * Hp + kk).ravel(), dyn // 4)
        if norm:
            # 1 / rms by wavefront tb over its staged row: KI * 8 reads a lane, or rms_inv_wave's over H
            check("gamma", np.arange(H), H)
            steps = KI * 8 if KI else -(-H // 64)
            rr = lane[:, None] + 64 * np.arange(steps)[None, :]
            rr = rr if KI else rr[rr < H]
            check("norm: a row's reads", np.ravel(rr), Hp)
            check("norm: s_x reads", (np.arange(nt)[:, None] * Hp + np.ravel(rr)[None, :]).ravel(), dyn // 4)
            check("s_r", np.arange(nt), TB)
        if xsplit:
            kh = np.arange(H)[None, :]
            check("xsplit", np.concatenate([((t0 + tb) * 2 * H + kh).ravel(),
                                            ((t0 + tb) * 2 * H + H + kh).ravel()]), T * 2 * H)
        # router weights (uint4 units): the first expert's (TB == 1) and the pair loads
        if KI:
            w_u4 = E * nq * 64
            if TB == 1:
                wv = np.arange(min(nw, E))[:, None, None]
                check("router w (first)", (wv * nq * 64 + lane[None, :, None] + 64 * np.arange(KI)[None, None, :]).ravel(), w_u4)
            e = np.arange(0, E, 1)[:, None]                  # every e some wavefront takes
            e1 = np.minimum(e + nw, E - 1)
            q = 64 * np.arange(KI)[None, :]
            check("router w (pair)", np.concatenate([(e * nq * 64 + q).ravel(), (e1 * nq * 64 + q + 63).ravel()]), w_u4)
            xs = lane[:, None] + 64 * (8 * np.arange(KI)[None, :, None] + np.arange(8)[None, None, :]).reshape(1, -1)
            check("router x reads", xs.ravel(), Hp)
        check("s_logit", [(nt - 1) * K_MAX_EXPERTS + E - 1], TB * K_MAX_EXPERTS)
        # activation records: a lane per 32-value block (write_records)
        nrec = 4 * -(-H // 128) if rec_terms == K_FINE_TERMS else 4 * K_GEMM_NS
        u = np.arange(nt * nrec)
        rtb, blk = u // nrec, u % nrec
        k0 = 32 * blk
        rd = (rtb * Hp)[:, None] + k0[:, None] + 4 * np.arange(8)[None, :]
        ok = (k0[:, None] + 4 * np.arange(8)[None, :] + 3) < Hp
        check("records: staging reads", (rd + 3)[ok], dyn // 4)
        spans = np.array([rec_offsets(rec_terms, int(x_)) for x_ in range(nrec)])  # [blk][n][2]
        lo = (t0 + rtb)[:, None] * rec_bytes + spans[blk][:, :, 0]
        hi = (t0 + rtb)[:, None] * rec_bytes + spans[blk][:, :, 1] - 1
        check("xrec", np.concatenate([lo.ravel(), hi.ravel()]), T * rec_bytes)
        # top-k stores
        t = t0 + np.arange(nt)[:, None]
        if per_wave:
            le = np.concatenate([lane[lane < E], lane[lane + 64 < E] + 64])
            check("logits", (t * E + le[None, :]).ravel(), T * E)
            check("s_logit top-k reads", le, K_MAX_EXPERTS)
        else:
            check("logits", (t * E + np.arange(E)[None, :]).ravel(), T * E)
        check("idx / wts", (t * k + np.arange(k)[None, :]).ravel(), N)
        # per-block counts and ranks (the table path's wavefront 0)
        ent = order[t0:t0 + nt].ravel()
        l = np.arange(nt * k)
        for j_, e_ in enumerate(ent):
            rank[t0 * k + j_] = blk_count[b, e_]
            blk_count[b, e_] += 1
        check("rank", t0 * k + l, N)
        check("blk_count", b * E + np.arange(E), T * E)
        if stamps:
            check("rt_ts stamps", b * 16 + np.array([0, 1, 3, 4, 5, 6, 9]), RT_STAMPS)
    # the last block: the count table in the x staging area, expert-major rows ld_bc apart
    # where route_bucket_fits; else k_bucket groups the entries in a launch of its own
    ld_bc = grid + 1
    fused = 18 * E <= Hp
    table = fused and ld_bc * E + 2 * E <= TB * Hp
    if table:
        i = np.arange(grid * E)
        bi = i // E
        check("s_bc fill", (i - bi * E) * ld_bc + bi, ld_bc * E)
        check("s_tot / s_base", ld_bc * E + np.arange(2 * E), dyn // 4)
        pref = np.zeros((E, grid), np.int64)               # exclusive prefix over blocks
        pref[:, 1:] = np.cumsum(blk_count.T, axis=1)[:, :-1]
        tot = blk_count.sum(axis=0)
        base = np.concatenate([[0], np.cumsum(tot)[:-1]])  # expert_list_wave: expert id order
        n = np.arange(N)
        e = order.ravel()
        ge = base[e] + pref[e, (n // k) // TB] + rank
        check("entry_src / pos scatter", ge, N)
        assert np.array_equal(np.sort(ge), n), "the scatter writes every entry exactly once"
        # entries of one expert ordered by t k + slot
        for ex in range(E):
            sel = np.nonzero(e == ex)[0]
            assert np.all(np.diff(ge[sel]) == 1)
    elif fused:
        # bucket_block in the staging area: (2 + 16) E ints
        check("bucket_block", np.arange(18 * E), dyn // 4)
    return dict(TB=TB, grid=grid, table=table, dyn=dyn)


@pytest.mark.parametrize("T,E,k", [(1, 32, 4), (2, 32, 4), (64, 32, 4), (2053, 32, 4), (4096, 32, 4),
                                   (2048, 128, 4), (64, 128, 4), (37, 32, 16), (2048, 32, 1)])
def test_route_indices_in_bounds(T, E, k):
    assert 18 * E <= 3072  # route_bucket_fits
    replay(T, E, k, 2880, rec_terms=3, xsplit=T < 64, seed=T + E)


@pytest.mark.parametrize("T,E,k,H,terms", [(7, 32, 4, 2880, 6), (64, 128, 4, 2880, 6), (3, 8, 2, 32, 6), (40, 64, 2, 1568, 6),
                                           (1, 32, 4, 3072, 6), (333, 16, 4, 2048, 3), (700, 40, 8, 544, 1), (2053, 40, 8, 2048, 3),
                                           (2053, 128, 4, 256, 1), (2050, 200, 3, 1024, 3)])
def test_route_norm_and_record_forms_in_bounds(T, E, k, H, terms):
    """The block forward's router (the norm's passes) and the records of 6 terms, of H's steps only."""
    for norm in (False, True):
        replay(T, E, k, H, rec_terms=terms, xsplit=T * k < 4 * E and terms == 3, seed=T + H, norm=norm)


RW_TOKENS, RW_THREADS, RW_MAIN, RW_MAX_E, RW_MAX_K = 16, 768, 512, 32, 4  # route_wide.hip: kRw*
RW_XROW, RW_WROW = 516, 65      # route_wide.hip: kRwXRow (floats), kRwWRow (uint4)
GRP_THREADS, GRP_BLOCKS = 1024, 8  # route_wide.hip: kGrpThreads, kGrpBlocks


def replay_wide(T, E, k, H, rec_terms=3, norm=False, seed=0, dropped=0.0):
    """k_route_wide's indices per workgroup, then k_group's on its ranks and counts; a share `dropped` of
    the entries has no expert (adaptive top-k)."""
    assert E <= RW_MAX_E and k <= RW_MAX_K and H % 32 == 0 and H <= 128 * K_GEMM_NS  # route_wide_fits
    nq = ((H + 63) // 64 + 7) // 8
    Hp, grid, N = nq * 512, -(-T // RW_TOKENS), T * k
    x_floats = RW_TOKENS * RW_XROW
    lds = x_floats * 4 + 32 * RW_WROW * 16
    static = 4 * (RW_TOKENS * RW_MAX_E + 2 * RW_TOKENS * K_MAX_TOPK + 2 * RW_TOKENS + RW_MAX_E)
    assert lds + static <= LDS_BYTES
    rec_bytes = row_bytes(rec_terms, H)
    tid = np.arange(RW_THREADS)
    lane, wv = tid & 63, tid >> 6
    m, lm, wm = tid[:RW_MAIN], lane[:RW_MAIN], wv[:RW_MAIN]
    sk, sr = 4 * (m & 127), m >> 7
    i4 = np.arange(4)[:, None]
    # staging writes of both tiles, each once
    xw = (4 * i4 + sr) * RW_XROW + sk
    assert np.unique((xw[..., None] + np.arange(4)).ravel()).size == RW_TOKENS * 512
    check("s_x tile", xw + 3, x_floats)
    ww = (8 * i4 + wm) * RW_WROW + lm
    assert np.unique(ww).size == 32 * 64
    check("s_wt tile", ww, 32 * RW_WROW)
    assert np.all(xw % 4 == 0) and (x_floats * 4) % 16 == 0  # 16-byte accesses
    # MFMA operands: residues res0 .. res0 + 3 of 16 experts and 16 tokens, steps h
    rs, es, col, blk = wm & 3, wm >> 2, lm & 15, lm >> 4
    res0 = 16 * rs + 4 * blk
    check("s_wt reads", (16 * es + col) * RW_WROW + res0 + i4, 32 * RW_WROW)
    check("s_x reads", col * RW_XROW + 64 * np.arange(8)[:, None] + res0 + 3, x_floats)
    # the exchange across the residue sets: [es][slot][8][lane] of f32x4 in the tiles' place
    slots = np.array([0, 1])
    check("s_ex", ((es[None, :] * 2 + slots[:, None]) * 8 + 7) * 64 + lm, lds // 16)
    e = 16 * es + 4 * blk + i4
    check("s_logit", col * RW_MAX_E + e[e < RW_MAX_E].max(), RW_TOKENS * RW_MAX_E)
    rng = np.random.default_rng(seed)
    order = np.argsort(rng.random((T, E)), axis=1)[:, :k].astype(np.int64)
    order[rng.random((T, k)) < dropped] = -1
    blk_count, rank = np.zeros((grid, E), np.int64), np.full(N, -1, np.int64)
    u = tid[RW_MAIN:] - RW_MAIN
    utb, ub = (u >> 2) & 15, (u & 3) + 4 * (u >> 6)
    check("record lanes' s_x reads", utb * RW_XROW + 32 * ub + 31, x_floats)
    spans = np.array([rec_offsets(rec_terms, b) for b in range(4 * K_GEMM_NS)])
    for b in range(grid):
        t0 = b * RW_TOKENS
        nt = min(RW_TOKENS, T - t0)
        if norm:
            row = t0 + np.minimum(np.arange(8)[:, None] + 8 * np.arange(2)[None, :], nt - 1)
            check("norm x", row.ravel() * H + H - 1, T * H)  # columns are min(k, H - 1)
            check("s_r", np.minimum(4 * i4 + sr, nt - 1), RW_TOKENS)
        done = np.zeros((nt, 4 * K_GEMM_NS), np.int64)
        for q in range(nq):
            kk = np.minimum(512 * q + sk, H - 4)
            row = t0 + np.minimum(4 * i4 + sr, nt - 1)
            check("x", row * H + kk + 3, T * H)
            check("gamma", kk + 3, H)
            check("router w", (np.minimum(8 * i4 + wm, E - 1) * nq + q) * 64 + lm, E * nq * 64)
            ok = (utb < nt) & (16 * q + ub < 4 * K_GEMM_NS)
            np.add.at(done, (utb[ok], 16 * q + ub[ok]), 1)
        b0 = 16 * nq
        nb = max(4 * K_GEMM_NS - b0, 0)
        z = np.arange(nt * nb)
        if nb:
            np.add.at(done, (z // nb, b0 + z - z // nb * nb), 1)
        assert np.all(done == 1), "every record block written once"
        rtb, rblk = np.nonzero(done)
        check("xrec", ((t0 + rtb)[:, None] * rec_bytes + spans[rblk][:, :, 1] - 1).ravel(), T * rec_bytes)
        check("logits", (t0 + nt - 1) * E + E - 1, T * E)
        ent = order[t0:t0 + nt].ravel()
        assert ent.size <= 64  # a lane per entry
        for j, ex in enumerate(ent):
            if ex >= 0:
                rank[t0 * k + j] = blk_count[b, ex]
                blk_count[b, ex] += 1
        check("blk_count", b * E + np.arange(E), T * E)
        check("rank", t0 * k + np.arange(ent.size), N)
    # k_group
    assert GRP_BLOCKS * RW_TOKENS * k <= GRP_THREADS
    P = GRP_THREADS // E
    tid = np.arange(GRP_THREADS)
    check("s_all", (P - 1) * E + E - 1, GRP_THREADS)
    tot = blk_count.sum(axis=0)
    base = np.concatenate([[0], np.cumsum(tot)[:-1]])
    ge = np.full(N, -1, np.int64)
    for g in range(-(-grid // GRP_BLOCKS)):
        b0 = g * GRP_BLOCKS
        seen = np.zeros(grid, np.int64)  # the table's rows, by part: r0 + i P
        for part in range(P):
            for r0 in range(part, grid, 8 * P):
                r = r0 + P * np.arange(8)
                np.add.at(seen, r[r < grid], 1)
        assert np.all(seen == 1)
        pre = [blk_count[:min(b0 + i, grid)].sum(axis=0) for i in range(GRP_BLOCKS)]
        n = b0 * RW_TOKENS * k + tid
        ok = (tid < GRP_BLOCKS * RW_TOKENS * k) & (n < N)
        for t, n_ in zip(tid[ok], n[ok]):
            ex = order.ravel()[n_]
            i = t // (RW_TOKENS * k)
            check("s_pre", i, GRP_BLOCKS)
            if ex >= 0:
                ge[n_] = base[ex] + pre[i][ex] + rank[n_]
    have = order.ravel() >= 0
    check("entry_src", ge[have], N)
    assert np.array_equal(np.sort(ge[have]), np.arange(have.sum())), "every entry lands exactly once"
    for ex in range(E):
        assert np.all(np.diff(ge[order.ravel() == ex]) == 1)
    return lds


@pytest.mark.parametrize("T,E,k,H,terms,dropped", [(896, 32, 4, 2880, 3, 0.0), (1025, 2, 1, 32, 3, 0.0), (1040, 3, 2, 96, 1, 0.0),
                                                   (1129, 17, 4, 544, 3, 0.3), (2049, 32, 4, 3072, 1, 0.0), (4096, 31, 3, 2048, 3, 0.5),
                                                   (897, 16, 1, 512, 3, 0.0)])
def test_wide_route_indices_in_bounds(T, E, k, H, terms, dropped):
    for norm in (False, True):
        replay_wide(T, E, k, H, rec_terms=terms, norm=norm, seed=T + E, dropped=dropped)


def test_route_trace_copy_configuration():
    """The configuration of the realtime-stamp trace copy: T = 4096, E = 32, k = 4 on the 20B
    shape, TB = 8, grid 512, dynamic LDS 8 Hp floats, the count table in the staging area; every
    index of the kernel and of the stamps in bounds, for both record forms."""
    for terms in (3, 1):
        r = replay(4096, 32, 4, 2880, rec_terms=terms, xsplit=False, seed=4096 + terms, stamps=True)
        assert (r["TB"], r["grid"], r["table"], r["dyn"]) == (8, 512, True, 8 * 3072 * 4)


def test_route_replay_detects_a_planted_overflow():
    """The replay's checks fire: a staging row one float longer than the launch's dynamic LDS."""
    with pytest.raises(AssertionError, match="s_x staging"):
        check("s_x staging", np.arange(8 * 3072 + 1), 8 * 3072)
