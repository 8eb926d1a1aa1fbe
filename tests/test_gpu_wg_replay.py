"""The anti-replay windows of bnk_wg_decap_batch (RFC 6479 as wireguard-go's
replay.Filter, one per peer, on the device, a whole batch at a time) against
the sequential filter of the oracle (bnko_replay_validate) fed packet by
packet in batch order, with wireguard-go's ordering: every authentic packet
goes through its peer's window before its inner header counts.  The window
itself is pinned on the CPU (tests/cpp/replay_test.cpp, tests/test_oracle_wg.py);
like the rest of the framing it is spec-derived, not a reference artefact."""
import struct

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P = 6
LIMIT = (1 << 64) - (1 << 13) - 1
WINDOW = 8128


def _peers():
    tx = [(1000 + 13 * i, 7000 + 17 * i, 0x64400001 + i, 0xFFFFFFFF) for i in range(P)]
    rx = [(p[1], p[0], p[2], p[3]) for p in tx]
    return tx, rx


def _inner(rng, src, length, kind):
    if kind == "keepalive":
        return b""
    pkt = bytearray(rng.integers(0, 256, length, dtype=np.uint8).tobytes())
    pkt[0] = 0x45 if kind != "badip" else 0x15
    pkt[2:4] = struct.pack(">H", length)
    pkt[12:16] = struct.pack(">I", src if kind != "notallowed" else src ^ 0x00010000)
    return bytes(pkt)


def _counters(rng, n, last):
    """A walk around each peer's newest counter: forward steps, repeats,
    reordering, the window's edges on both sides, far jumps."""
    peer = rng.integers(0, P, n)
    ctr = np.zeros(n, np.uint64)
    last = list(last)
    recent = [[] for _ in range(P)]
    for i in range(n):
        p = int(peer[i])
        r = rng.random()
        if r < 0.55:
            c = last[p] + int(rng.integers(1, 4))
        elif r < 0.70 and recent[p]:
            c = recent[p][int(rng.integers(0, len(recent[p])))]          # an exact repeat
        elif r < 0.80:
            c = max(0, last[p] - int(rng.integers(0, 200)))              # a little late
        elif r < 0.86:
            c = max(0, last[p] - WINDOW + int(rng.integers(-2, 3)))      # the far edge of the window
        elif r < 0.90:
            c = last[p] + int(rng.integers(60, 70)) * int(rng.integers(1, 200))  # over one or many blocks
        elif r < 0.93:
            c = last[p] + WINDOW + int(rng.integers(-2, 3)) + 64         # just beyond a whole ring
        elif r < 0.95:
            c = 0
        else:
            c = last[p] + int(rng.integers(1, 3))
        c = min(c, LIMIT + 3)
        ctr[i] = c
        if c < LIMIT:
            last[p] = max(last[p], c)
        recent[p] = (recent[p] + [c])[-50:]
    return peer.astype(np.uint32), ctr, last


def _batch(rng, tx, keys, n, last, near_limit=False):
    from oracle import binding as O
    peer, ctr, last = _counters(rng, n, last)
    if near_limit:
        ctr[:6] = np.array([LIMIT - 2, LIMIT - 1, LIMIT, LIMIT + 1, LIMIT - 1, LIMIT - 2], np.uint64)
        peer[:6] = 0
    kinds = rng.choice(["ok", "ok", "ok", "ok", "keepalive", "notallowed", "badip", "forged"], n)
    wires, offs, pos = [], np.zeros(n, np.uint64), 0
    for i in range(n):
        p = int(peer[i])
        inner = _inner(rng, tx[p][2], int(rng.choice([20, 28, 60, 200, 576])), kinds[i])
        w = bytearray(O.wg_encap(inner, 1420, keys[p].tobytes(), tx[p][1], int(ctr[i])))
        if kinds[i] == "forged":
            w[-1] ^= 1
        offs[i] = pos
        wires.append(bytes(w))
        pos += (len(w) + 15) & ~15
    arena = np.zeros(pos + 16, np.uint8)
    for i, w in enumerate(wires):
        arena[int(offs[i]):int(offs[i]) + len(w)] = np.frombuffer(w, np.uint8)
    lens = np.array([len(w) for w in wires], np.uint32)
    return arena, offs, lens, wires, last


def _expect(wires, rx, keys, filters):
    """Oracle result per packet, then the sequential window per peer in batch order."""
    from bnk_amd import lib
    from oracle import binding as O
    n = len(wires)
    res, olen, peer, ctr = np.zeros(n, np.uint8), np.zeros(n, np.uint32), np.zeros(n, np.uint32), np.zeros(n, np.uint64)
    for i, w in enumerate(wires):
        rc, pt, p, c = O.wg_decap(w, rx, keys)
        res[i], olen[i], peer[i], ctr[i] = rc, len(pt), p, c
        if rc not in (lib.WG_BAD_HEADER, lib.WG_UNKNOWN_INDEX, lib.WG_AUTH_FAIL):
            if not filters[p].validate(c):
                res[i], olen[i] = lib.WG_REPLAY, 0
    return res, olen, peer, ctr


@pytest.mark.parametrize("mode", ["host_fused", "host_unfused", "device_large", "device_separate", "ring_fused",
                                  "device_block"])
def test_replay_windows_match_the_sequential_filter(mode):
    import torch
    from bnk_amd import lib
    from oracle import binding as O
    rng = np.random.default_rng(2024)
    tx, rx = _peers()
    keys = rng.integers(0, 256, (P, 32), dtype=np.uint8)
    filters = [O.ReplayFilter() for _ in range(P)]
    last = [0] * P
    sizes = {"host_fused": [1, 64, 300, 1024, 700], "host_unfused": [300, 1024, 2000, 150],
             "device_large": [5000, 1025, 9000, 3000], "device_separate": [3000, 1025, 6000],
             "ring_fused": [128, 900, 128], "device_block": [1025, 4096, 2047, 4097, 4095]}[mode]
    seen = set()
    with lib.Context(0) as ctx:
        ctx.keys_set(lib.KEYS_RECV, keys)
        ctx.wg_peers_set(rx)
        if mode == "host_unfused":
            ctx.set_spread_max_packets(0)
        if mode == "device_separate":
            ctx.wg_set_fused(False)  # the framing, and the window pass's sort keys, from kernels of their own
        for b, n in enumerate(sizes):
            arena, offs, lens, wires, last = _batch(rng, tx, keys, n, last, near_limit=(b == 2))
            want = _expect(wires, rx, keys, filters)
            total = arena.nbytes
            if mode.startswith("device"):
                d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")  # noqa: E731
                d_arena, d_out = d(arena), torch.zeros(total, dtype=torch.uint8, device="cuda:0")
                res = torch.zeros(n, dtype=torch.uint8, device="cuda:0")
                olen = torch.zeros(n, dtype=torch.int32, device="cuda:0")
                gp = torch.zeros(n, dtype=torch.int32, device="cuda:0")
                gc = torch.zeros(n, dtype=torch.int64, device="cuda:0")
                d_off, d_len = d(offs.astype(np.int64)), d(lens.astype(np.int32))
                torch.cuda.synchronize()
                ctx.wg_decap(lib.make_batch(d_arena, total, n, lib.MEM_DEVICE, offsets=d_off, lens=d_len),
                             lib.make_batch(d_out, total, n, lib.MEM_DEVICE, offsets=d_off), res, olen, gp, gc)
                ctx.sync()
                got = (res.cpu().numpy(), olen.cpu().numpy().astype(np.uint32), gp.cpu().numpy().astype(np.uint32),
                       gc.cpu().numpy().astype(np.uint64))
            else:
                rings = []
                if mode == "ring_fused":
                    rings = [ctx.ring_alloc(total), ctx.ring_alloc(total)]
                    rings[0][:] = arena
                src = rings[0] if rings else arena
                out = rings[1] if rings else np.zeros(total, np.uint8)
                res, olen = np.zeros(n, np.uint8), np.zeros(n, np.uint32)
                gp, gc = np.zeros(n, np.uint32), np.zeros(n, np.uint64)
                ctx.wg_decap(lib.make_batch(src, total, n, lib.MEM_HOST, offsets=offs, lens=lens),
                             lib.make_batch(out, total, n, lib.MEM_HOST, offsets=offs), res, olen, gp, gc)
                got = (res, olen, gp, gc)
                for r in rings:
                    ctx.ring_free(r)
            bad = np.flatnonzero(got[0] != want[0])
            assert bad.size == 0, f"batch {b}: result differs at {bad[:5]}: got {got[0][bad[:5]]} want {want[0][bad[:5]]}"
            assert np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2]) and np.array_equal(got[3], want[3])
            seen.update(np.unique(want[0]).tolist())
    # the walk exercised every outcome, replays among them
    assert {lib.WG_OK, lib.WG_KEEPALIVE, lib.WG_AUTH_FAIL, lib.WG_BAD_IP, lib.WG_NOT_ALLOWED, lib.WG_REPLAY} <= seen


def test_a_rekeyed_peer_starts_with_an_empty_window_and_the_switch_turns_windows_off():
    from bnk_amd import lib
    from oracle import binding as O
    rng = np.random.default_rng(7)
    tx, rx = _peers()
    keys = rng.integers(0, 256, (P, 32), dtype=np.uint8)

    def decap(ctx, wires):
        n = len(wires)
        offs = np.arange(n, dtype=np.uint64) * 128
        arena = np.zeros(n * 128, np.uint8)
        for i, w in enumerate(wires):
            arena[i * 128:i * 128 + len(w)] = np.frombuffer(w, np.uint8)
        lens = np.array([len(w) for w in wires], np.uint32)
        out = np.zeros_like(arena)
        res, olen, gp, gc = np.zeros(n, np.uint8), np.zeros(n, np.uint32), np.zeros(n, np.uint32), np.zeros(n, np.uint64)
        ctx.wg_decap(lib.make_batch(arena, arena.nbytes, n, lib.MEM_HOST, offsets=offs, lens=lens),
                     lib.make_batch(out, out.nbytes, n, lib.MEM_HOST, offsets=offs), res, olen, gp, gc)
        return res.tolist()

    def dg(p, c, key=None, remote=None):
        inner = _inner(rng, tx[p][2], 40, "ok")
        return O.wg_encap(inner, 1420, (keys[p] if key is None else key).tobytes(), tx[p][1] if remote is None else remote, c)

    with lib.Context(0) as ctx:
        ctx.keys_set(lib.KEYS_RECV, keys)
        ctx.wg_peers_set(rx)
        assert decap(ctx, [dg(0, 5), dg(1, 5), dg(0, 5), dg(0, 4)]) == [lib.WG_OK, lib.WG_OK, lib.WG_REPLAY, lib.WG_OK]
        assert decap(ctx, [dg(0, 5), dg(0, 4), dg(1, 5), dg(0, 6)]) == [lib.WG_REPLAY] * 3 + [lib.WG_OK]
        # peer 0 rekeys: new indices, new key, and a window that has seen nothing;
        # peer 1's window stands
        new_key = rng.integers(0, 256, 32, dtype=np.uint8)
        ctx.wg_peer_set(0, (rx[0][0] + 1, rx[0][1], rx[0][2], rx[0][3]), key_recv=new_key)
        assert decap(ctx, [dg(0, 5, new_key, rx[0][0] + 1), dg(1, 5), dg(0, 5)]) == \
            [lib.WG_OK, lib.WG_REPLAY, lib.WG_UNKNOWN_INDEX]
        # the same table again keeps the windows; a changed row starts over
        rows = [(rx[0][0] + 1, rx[0][1], rx[0][2], rx[0][3])] + rx[1:]
        ctx.wg_peers_set(rows)
        assert decap(ctx, [dg(0, 5, new_key, rx[0][0] + 1), dg(1, 5)]) == [lib.WG_REPLAY, lib.WG_REPLAY]
        rows[1] = (rx[1][0] + 1, rx[1][1], rx[1][2], rx[1][3])
        ctx.wg_peers_set(rows)
        assert decap(ctx, [dg(1, 5, None, rx[1][0] + 1), dg(0, 5, new_key, rx[0][0] + 1)]) == [lib.WG_OK, lib.WG_REPLAY]
        # windows off: nothing is turned away and nothing is recorded
        ctx.wg_set_replay(False)
        assert decap(ctx, [dg(2, 9), dg(2, 9)]) == [lib.WG_OK, lib.WG_OK]
        ctx.wg_set_replay(True)
        assert decap(ctx, [dg(2, 9), dg(2, 9)]) == [lib.WG_OK, lib.WG_REPLAY]


def _traffic(tx_ctx, tx_peers, n_a, n_b, n_total, inner_len, jump_rows, rng):
    """Datagrams for a large decapsulating batch without a per-packet oracle:
    two encapsulated batches (between them some peers' send counters jump ahead
    by more than a window, so that the first batch's packets of those peers are
    too old once a second-batch packet has been seen), then a shuffled mix of
    both with repeats.  Returns the wire arena, offsets, lengths, and each
    datagram's sender and counter as the sending side knows them."""
    from bnk_amd import lib
    n_peers = len(tx_peers)
    slot = (16 + inner_len + 15 + 16 + 15) & ~15
    per = []
    for k, n in enumerate((n_a, n_b)):
        peer = rng.integers(0, n_peers, n).astype(np.uint32)
        # half of either batch belongs to the peers that jump, so that they have old
        # packets to be refused and new ones to refuse them
        peer[: n // 2] = rng.choice(jump_rows, n // 2).astype(np.uint32)
        arena = rng.integers(0, 256, n * slot, dtype=np.uint8)
        rows = arena.reshape(n, slot)
        rows[:, 16] = 0x45
        rows[:, 18], rows[:, 19] = inner_len >> 8, inner_len & 255
        allowed = np.array([t[2] for t in tx_peers], np.uint32)[peer]
        rows[:, 28:32] = allowed.astype(">u4").view(np.uint8).reshape(n, 4)
        wl = np.zeros(n, np.uint32)
        if k == 1:
            for r in jump_rows:
                tx_ctx.wg_send_counter_set(int(r), 9000 + int(r) % 7)
        tx_ctx.wg_encap(lib.make_batch(arena, arena.nbytes, n, lib.MEM_HOST, stride=slot, length=inner_len,
                                       peer=peer), 1420, wl)
        assert (wl == 16 + ((inner_len + 15) & ~15) + 16).all()
        per.append((arena.reshape(n, slot), peer, int(wl[0])))
    wire_len = per[0][2]
    src = np.concatenate([per[0][0], per[1][0]])[:, :wire_len]
    src_peer = np.concatenate([per[0][1], per[1][1]])
    pick = np.concatenate([np.arange(n_a + n_b), rng.integers(0, n_a + n_b, n_total - n_a - n_b)])
    rng.shuffle(pick)
    stride = (wire_len + 15) & ~15
    wire = np.zeros((n_total, stride), np.uint8)
    wire[:, :wire_len] = src[pick]
    ctr = wire[:, 8:16].copy().view("<u8").reshape(-1)
    return wire.reshape(-1), stride, wire_len, src_peer[pick], ctr


def _window_expectation(peer, ctr, n_peers_seen):
    from bnk_amd import lib
    from oracle import binding as O
    filters = {}
    want = np.zeros(len(peer), np.uint8)
    for i in range(len(peer)):
        f = filters.setdefault(int(peer[i]), O.ReplayFilter())
        want[i] = lib.WG_OK if f.validate(int(ctr[i])) else lib.WG_REPLAY
    return want


def test_window_pass_with_more_peers_than_a_packed_sort_key_holds():
    """70,000 peers and 40,000 packets: the sender's number and the packet's
    position no longer fit one 32-bit sort key, so the window pass sorts
    (sender, position) pairs.  Expected results come from the sequential
    filter fed, in batch order, the senders and counters the sending side
    assigned."""
    import torch
    from bnk_amd import lib
    rng = np.random.default_rng(77)
    n_peers, n_total = 70000, 40000
    tx = [(10 + 3 * i, 500000 + 5 * i, 0x64400000 + i, 0xFFFFFFFF) for i in range(n_peers)]
    rx = [(p[1], p[0], p[2], p[3]) for p in tx]
    keys = rng.integers(0, 256, (n_peers, 32), dtype=np.uint8)
    jump_rows = rng.choice(n_peers, 300, replace=False)
    with lib.Context(0) as txc, lib.Context(0) as rxc:
        txc.keys_set(lib.KEYS_SEND, keys)
        txc.wg_peers_set(tx)
        rxc.keys_set(lib.KEYS_RECV, keys)
        rxc.wg_peers_set(rx)
        wire, stride, wire_len, peer, ctr = _traffic(txc, tx, 12000, 8000, n_total, 40, jump_rows, rng)
        want = _window_expectation(peer, ctr, n_peers)
        d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")  # noqa: E731
        d_wire, d_out = d(wire), torch.zeros(wire.nbytes, dtype=torch.uint8, device="cuda:0")
        res = torch.zeros(n_total, dtype=torch.uint8, device="cuda:0")
        olen = torch.zeros(n_total, dtype=torch.int32, device="cuda:0")
        gp = torch.zeros(n_total, dtype=torch.int32, device="cuda:0")
        gc = torch.zeros(n_total, dtype=torch.int64, device="cuda:0")
        torch.cuda.synchronize()
        rxc.wg_decap(lib.make_batch(d_wire, wire.nbytes, n_total, lib.MEM_DEVICE, stride=stride, length=wire_len),
                     lib.make_batch(d_out, wire.nbytes, n_total, lib.MEM_DEVICE, stride=stride), res, olen, gp, gc)
        rxc.sync()
        assert np.array_equal(gp.cpu().numpy().astype(np.uint32), peer)
        assert np.array_equal(gc.cpu().numpy().astype(np.uint64), ctr)
        got = res.cpu().numpy()
        bad = np.flatnonzero(got != want)
        assert bad.size == 0, f"result differs at {bad[:5]}: got {got[bad[:5]]} want {want[bad[:5]]}"
        assert (want == lib.WG_REPLAY).sum() > 1000 and (want == lib.WG_OK).sum() > 1000
        assert np.array_equal(olen.cpu().numpy() != 0, want == lib.WG_OK)


@pytest.mark.parametrize("n_peers,n_total", [(255, 66000), (2047, 66000), (2048, 66000), (3, 530000)])
def test_window_pass_sorted_by_counting_and_where_that_ends(n_peers, n_total):
    """A key more than there are peers fills the counting sort's row of 256 or the last of the
    rows it is used for, or goes beyond them; tiles of one run and of several, the last one
    ragged; some tags forged, so that packets without a sender take part."""
    import torch
    from bnk_amd import lib
    rng = np.random.default_rng(n_peers)
    tx = [(10 + 3 * i, 500000 + 5 * i, 0x64400000 + i, 0xFFFFFFFF) for i in range(n_peers)]
    rx = [(p[1], p[0], p[2], p[3]) for p in tx]
    keys = rng.integers(0, 256, (n_peers, 32), dtype=np.uint8)
    jump_rows = rng.choice(n_peers, max(1, n_peers // 8), replace=False)
    with lib.Context(0) as txc, lib.Context(0) as rxc:
        txc.keys_set(lib.KEYS_SEND, keys)
        txc.wg_peers_set(tx)
        rxc.keys_set(lib.KEYS_RECV, keys)
        rxc.wg_peers_set(rx)
        wire, stride, wire_len, peer, ctr = _traffic(txc, tx, n_total // 3, n_total // 5, n_total, 40, jump_rows, rng)
        forged = rng.choice(n_total, n_total // 50, replace=False)
        wire.reshape(-1)[forged.astype(np.int64) * stride + wire_len - 1] ^= 1
        good = np.ones(n_total, bool)
        good[forged] = False
        want = np.full(n_total, lib.WG_AUTH_FAIL, np.uint8)
        want[good] = _window_expectation(peer[good], ctr[good], n_peers)
        d_wire = torch.from_numpy(np.ascontiguousarray(wire)).to("cuda:0")
        d_out = torch.zeros(wire.nbytes, dtype=torch.uint8, device="cuda:0")
        res = torch.zeros(n_total, dtype=torch.uint8, device="cuda:0")
        olen, gp = (torch.zeros(n_total, dtype=torch.int32, device="cuda:0") for _ in range(2))
        gc = torch.zeros(n_total, dtype=torch.int64, device="cuda:0")
        torch.cuda.synchronize()
        rxc.wg_decap(lib.make_batch(d_wire, wire.nbytes, n_total, lib.MEM_DEVICE, stride=stride, length=wire_len),
                     lib.make_batch(d_out, wire.nbytes, n_total, lib.MEM_DEVICE, stride=stride), res, olen, gp, gc)
        rxc.sync()
        assert np.array_equal(gp.cpu().numpy().astype(np.uint32), peer)
        got = res.cpu().numpy()
        bad = np.flatnonzero(got != want)
        assert bad.size == 0, f"result differs at {bad[:5]}: got {got[bad[:5]]} want {want[bad[:5]]}"
        assert (want == lib.WG_REPLAY).sum() > 1000 and (want == lib.WG_OK).sum() > 1000


def test_window_pass_of_a_host_batch_that_goes_through_in_chunks():
    """A host batch beyond the size that runs in one piece is cut into chunks,
    each with a window pass of its own continuing the one before: results are
    those of the sequential filter over the whole batch in order."""
    from bnk_amd import lib
    rng = np.random.default_rng(78)
    n_peers, n_total = 40, 14000
    tx = [(100 + 3 * i, 9000 + 5 * i, 0x64400000 + i, 0xFFFFFFFF) for i in range(n_peers)]
    rx = [(p[1], p[0], p[2], p[3]) for p in tx]
    keys = rng.integers(0, 256, (n_peers, 32), dtype=np.uint8)
    with lib.Context(0) as txc, lib.Context(0) as rxc:
        txc.keys_set(lib.KEYS_SEND, keys)
        txc.wg_peers_set(tx)
        rxc.keys_set(lib.KEYS_RECV, keys)
        rxc.wg_peers_set(rx)
        wire, stride, wire_len, peer, ctr = _traffic(txc, tx, 6000, 5000, n_total, 1400, np.arange(0, n_peers, 3),
                                                     rng)
        assert wire.nbytes > (16 << 20)  # well beyond two chunks' worth
        want = _window_expectation(peer, ctr, n_peers)
        out = np.zeros(wire.nbytes, np.uint8)
        res, olen = np.zeros(n_total, np.uint8), np.zeros(n_total, np.uint32)
        gp, gc = np.zeros(n_total, np.uint32), np.zeros(n_total, np.uint64)
        rxc.wg_decap(lib.make_batch(wire, wire.nbytes, n_total, lib.MEM_HOST, stride=stride, length=wire_len),
                     lib.make_batch(out, out.nbytes, n_total, lib.MEM_HOST, stride=stride), res, olen, gp, gc)
        assert np.array_equal(gp, peer) and np.array_equal(gc, ctr)
        bad = np.flatnonzero(res != want)
        assert bad.size == 0, f"result differs at {bad[:5]}: got {res[bad[:5]]} want {want[bad[:5]]}"
        assert (want == lib.WG_REPLAY).sum() > 1000 and (want == lib.WG_OK).sum() > 1000


def test_window_pass_where_one_peer_fills_more_blocks_than_one_look_back_reads():
    """Two peers, one of them sending nearly everything: its run in sorted order
    spans well over a thousand blocks of 1024 positions, so the running maximum
    a block is handed comes from carries read in more than one step, and a late
    repeat of a counter that was ahead when it first came is found by a search
    that goes back across many blocks."""
    import torch
    from bnk_amd import lib
    rng = np.random.default_rng(79)
    n_total = 2_300_000
    tx = [(100, 9000, 0x64400000, 0xFFFFFFFF), (103, 9005, 0x64400001, 0xFFFFFFFF)]
    rx = [(p[1], p[0], p[2], p[3]) for p in tx]
    keys = rng.integers(0, 256, (2, 32), dtype=np.uint8)
    with lib.Context(0) as txc, lib.Context(0) as rxc:
        txc.keys_set(lib.KEYS_SEND, keys)
        txc.wg_peers_set(tx)
        rxc.keys_set(lib.KEYS_RECV, keys)
        rxc.wg_peers_set(rx)
        # (no jump: a window is far shorter than the batch, so most early packets are too old
        # by the time they come, the rest repeat or are fresh)
        wire, stride, wire_len, peer, ctr = _traffic(txc, tx, 700_000, 500_000, n_total, 40, np.array([0]), rng)
        # the first 1.2 million in sending order, so that long stretches are ahead of everything
        # before them, then the shuffled mix with its repeats
        order = np.argsort(ctr[:1_200_000], kind="stable")
        w2 = wire.reshape(n_total, stride)
        w2[:1_200_000] = w2[:1_200_000][order]
        peer[:1_200_000], ctr[:1_200_000] = peer[:1_200_000][order], ctr[:1_200_000][order]
        assert (peer == 0).sum() > 1_500_000
        want = _window_expectation(peer, ctr, 2)
        d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")  # noqa: E731
        d_wire, d_out = d(wire), torch.zeros(wire.nbytes, dtype=torch.uint8, device="cuda:0")
        res = torch.zeros(n_total, dtype=torch.uint8, device="cuda:0")
        olen = torch.zeros(n_total, dtype=torch.int32, device="cuda:0")
        gp = torch.zeros(n_total, dtype=torch.int32, device="cuda:0")
        gc = torch.zeros(n_total, dtype=torch.int64, device="cuda:0")
        torch.cuda.synchronize()
        rxc.wg_decap(lib.make_batch(d_wire, wire.nbytes, n_total, lib.MEM_DEVICE, stride=stride, length=wire_len),
                     lib.make_batch(d_out, wire.nbytes, n_total, lib.MEM_DEVICE, stride=stride), res, olen, gp, gc)
        rxc.sync()
        assert np.array_equal(gp.cpu().numpy().astype(np.uint32), peer)
        assert np.array_equal(gc.cpu().numpy().astype(np.uint64), ctr)
        got = res.cpu().numpy()
        bad = np.flatnonzero(got != want)
        assert bad.size == 0, f"result differs at {bad[:5]}: got {got[bad[:5]]} want {want[bad[:5]]}"
        assert (want == lib.WG_REPLAY).sum() > 100_000 and (want == lib.WG_OK).sum() > 100_000
        # the same datagrams again: the windows have seen or passed every counter
        rxc.wg_decap(lib.make_batch(d_wire, wire.nbytes, n_total, lib.MEM_DEVICE, stride=stride, length=wire_len),
                     lib.make_batch(d_out, wire.nbytes, n_total, lib.MEM_DEVICE, stride=stride), res, olen, gp, gc)
        rxc.sync()
        assert (res.cpu().numpy() == lib.WG_REPLAY).all()


@pytest.mark.parametrize("peers", [1, 2, 40])
def test_window_pass_with_few_and_many_senders(peers, monkeypatch):
    """The same walk as above, device resident, with one sender (every run spans
    several blocks of the pass, so repeats are looked for across blocks and a
    block's running maximum comes from the blocks before it), two, and forty
    (short runs, several to a block), per packet against the sequential filter."""
    import torch
    import sys
    from bnk_amd import lib
    from oracle import binding as O
    monkeypatch.setattr(sys.modules[__name__], "P", peers)
    rng = np.random.default_rng(300 + peers)
    tx, rx = _peers()
    keys = rng.integers(0, 256, (peers, 32), dtype=np.uint8)
    filters = [O.ReplayFilter() for _ in range(peers)]
    last = [0] * peers
    with lib.Context(0) as ctx:
        ctx.keys_set(lib.KEYS_RECV, keys)
        ctx.wg_peers_set(rx)
        for b, n in enumerate([3000, 1100, 6000, 2500]):
            arena, offs, lens, wires, last = _batch(rng, tx, keys, n, last, near_limit=(b == 1))
            want = _expect(wires, rx, keys, filters)
            total = arena.nbytes
            d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")  # noqa: E731
            d_arena, d_out = d(arena), torch.zeros(total, dtype=torch.uint8, device="cuda:0")
            res = torch.zeros(n, dtype=torch.uint8, device="cuda:0")
            olen = torch.zeros(n, dtype=torch.int32, device="cuda:0")
            gp = torch.zeros(n, dtype=torch.int32, device="cuda:0")
            gc = torch.zeros(n, dtype=torch.int64, device="cuda:0")
            d_off, d_len = d(offs.astype(np.int64)), d(lens.astype(np.int32))
            torch.cuda.synchronize()
            ctx.wg_decap(lib.make_batch(d_arena, total, n, lib.MEM_DEVICE, offsets=d_off, lens=d_len),
                         lib.make_batch(d_out, total, n, lib.MEM_DEVICE, offsets=d_off), res, olen, gp, gc)
            ctx.sync()
            got = res.cpu().numpy()
            bad = np.flatnonzero(got != want[0])
            assert bad.size == 0, f"batch {b}: result differs at {bad[:5]}: got {got[bad[:5]]} want {want[0][bad[:5]]}"
            assert np.array_equal(olen.cpu().numpy().astype(np.uint32), want[1])
            assert (want[0] == lib.WG_REPLAY).sum() > 50


@pytest.mark.parametrize("n_peers,n", [(1, 1025), (2, 4096), (127, 4095), (254, 4096), (255, 3000), (256, 4096),
                                       (4097, 2048), (65534, 4096), (70000, 1026)])
def test_counters_and_windows_of_one_workgroup_over_the_peers_digits(n_peers, n):
    """1025 to 4096 packets take their send counters and go through their windows in one
    workgroup each, sorted by sender eight bits at a time at most: tables of one, two and three
    passes and their edges, counters against the count of earlier packets of the peer, windows
    (repeats, old packets, jumps) against the sequential filter."""
    import torch
    from bnk_amd import lib
    from oracle import binding as O
    rng = np.random.default_rng(n_peers + n)
    tx = [(10 + 3 * i, 500000 + 5 * i, 0x64400000 + i, 0xFFFFFFFF) for i in range(n_peers)]
    rx = [(p[1], p[0], p[2], p[3]) for p in tx]
    keys = rng.integers(0, 256, (n_peers, 32), dtype=np.uint8)
    # the table's ends, a crowd at one of them and everything between
    peer = rng.integers(0, n_peers, n).astype(np.uint32)
    peer[:n // 4] = n_peers - 1
    peer[n // 4:n // 3] = rng.integers(0, min(n_peers, 5), n // 3 - n // 4)
    rng.shuffle(peer)
    slot, length = 96, 40
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")  # noqa: E731
    with lib.Context(0) as txc, lib.Context(0) as rxc:
        txc.keys_set(lib.KEYS_SEND, keys)
        txc.wg_peers_set(tx)
        rxc.keys_set(lib.KEYS_RECV, keys)
        rxc.wg_peers_set(rx)
        first = {int(p): 9000 + int(p) % 7 for p in rng.choice(n_peers, min(n_peers, 40), replace=False)}
        for p, c in first.items():
            txc.wg_send_counter_set(p, c)
        wires, ctrs, nxt = [], [], np.array([first.get(p, 0) for p in range(n_peers)], np.uint64)
        for _ in range(2):
            rows = rng.integers(0, 256, (n, slot), dtype=np.uint8)
            rows[:, 16], rows[:, 18], rows[:, 19] = 0x45, 0, length
            rows[:, 28:32] = np.array([t[2] for t in tx], np.uint32)[peer].astype(">u4").view(np.uint8).reshape(n, 4)
            want = np.zeros(n, np.uint64)
            for i in range(n):
                want[i] = nxt[peer[i]]
                nxt[peer[i]] += 1
            buf, wl = d(rows.reshape(-1)), torch.zeros(n, dtype=torch.int32, device="cuda:0")
            torch.cuda.synchronize()
            txc.wg_encap(lib.make_batch(buf, n * slot, n, lib.MEM_DEVICE, stride=slot, length=length, peer=d(peer.view(np.int32))), 1420, wl)
            txc.sync()
            assert (wl == 80).all()
            wires.append(buf.cpu().numpy().reshape(n, slot))
            got = wires[-1][:, 8:16].copy().view("<u8").reshape(-1)
            assert np.array_equal(got, want)
            ctrs.append(want)
        assert np.array_equal(txc.wg_send_counters(n_peers), nxt)
        # one batch of each half and of both again, in any order
        both, who, ctr = np.concatenate(wires), np.concatenate([peer, peer]), np.concatenate(ctrs)
        filters = {}
        for _ in range(2):
            pick = rng.integers(0, 2 * n, n)
            want = np.array([lib.WG_OK if filters.setdefault(int(who[i]), O.ReplayFilter()).validate(int(ctr[i])) else lib.WG_REPLAY
                             for i in pick], np.uint8)
            wire, out = d(both[pick].reshape(-1)), torch.zeros(n * slot, dtype=torch.uint8, device="cuda:0")
            res = torch.full((n,), 99, dtype=torch.uint8, device="cuda:0")
            olen, gp = (torch.zeros(n, dtype=torch.int32, device="cuda:0") for _ in range(2))
            gc = torch.zeros(n, dtype=torch.int64, device="cuda:0")
            torch.cuda.synchronize()
            rxc.wg_decap(lib.make_batch(wire, n * slot, n, lib.MEM_DEVICE, stride=slot, length=80),
                         lib.make_batch(out, n * slot, n, lib.MEM_DEVICE, stride=slot), res, olen, gp, gc)
            rxc.sync()
            assert np.array_equal(gc.cpu().numpy().view(np.uint64), ctr[pick])
            assert np.array_equal(res.cpu().numpy(), want)
            assert np.array_equal(olen.cpu().numpy(), np.where(want == lib.WG_OK, length, 0))
            assert len(np.unique(want)) == 2


@pytest.mark.parametrize("n_peers,n", [(1, 4097), (255, 5000), (256, 8191), (1023, 32768), (1024, 6000), (3, 32769)])
def test_tunnel_batches_whose_tiles_add_up_the_rows_before_theirs(n_peers, n):
    """NoteOutbound and encapsulation, then decapsulation, windows and CheckInbound of device-resident
    batches between those of one workgroup and those with a launch for the scan: tables of one row of
    columns, of several and of one key too many, batches of one run a tile and of as many as a wave
    keeps; counters against the count of earlier packets, windows (repeats, old packets, jumps, two
    batches in a row) against the sequential filter, verdicts and the flow tables against the oracle."""
    import torch
    from bnk_amd import lib
    from bnk_amd import workloads as W
    from oracle import binding as O
    rng = np.random.default_rng(n_peers + n)
    base, t0 = 0x64400000, 1_700_000_000 * 10**9
    tx = [(10 + 3 * i, 500000 + 5 * i, base + i, 0xFFFFFFFF) for i in range(n_peers)]
    rx = [(p[1], p[0], p[2], p[3]) for p in tx]
    keys = rng.integers(0, 256, (n_peers, 32), dtype=np.uint8)
    rules = [([(base, 10)], "tcp", [(0, 999)]), ([(base, 10)], "udp", [(65000, 65535)])]
    peer = rng.integers(0, n_peers, n).astype(np.uint32)
    peer[:n // 3] = n_peers - 1
    rng.shuffle(peer)
    slot, length = 96, 40
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")  # noqa: E731
    i32 = lambda: torch.full((n,), 99, dtype=torch.int32, device="cuda:0")  # noqa: E731
    at = lambda m: (np.arange(m, dtype=np.uint64) * slot, np.full(m, length, np.uint32))  # noqa: E731
    with lib.Context(0) as txc, lib.Context(0) as rxc:
        sent, flows_in = O.Filter(), O.Filter()
        for c, o, k in ((txc, sent, lib.KEYS_SEND), (rxc, flows_in, lib.KEYS_RECV)):
            c.keys_set(k, keys)
            c.wg_peers_set(tx if c is txc else rx)
            c.filter_set_rules(rules)
            o.set_rules(rules)
        first = {int(p): 9000 + int(p) % 7 for p in rng.choice(n_peers, min(n_peers, 40), replace=False)}
        for p, c in first.items():
            txc.wg_send_counter_set(p, c)
        nxt = np.array([first.get(p, 0) for p in range(n_peers)], np.uint64)
        wires, inner, ctrs = [], [], []
        for k in range(2):
            src = (base + peer).astype(np.uint32)
            proto = rng.choice([6, 17, 1], n).astype(np.uint8)
            rec = W.header_records(proto, src, np.full(n, base | 0xFFFF, np.uint32), rng.integers(0, 2000, n).astype(np.uint32),
                                   rng.choice([0, 999, 1000, 64999, 65000, 65535], n).astype(np.uint32))
            rows = rng.integers(0, 256, (n, slot), dtype=np.uint8)
            rows[:, 16:16 + 28] = rec[:, :28]
            rows[:, 18], rows[:, 19] = 0, length
            want = np.zeros(n, np.uint64)
            for i in range(n):
                want[i] = nxt[peer[i]]
                nxt[peer[i]] += 1
            sent.note_outbound_batch(np.ascontiguousarray(rows[:, 16:]).reshape(-1), np.arange(n, dtype=np.uint64) * (slot - 16),
                                     at(n)[1], t0 + k)
            buf, wl = d(rows.reshape(-1)), i32()
            torch.cuda.synchronize()
            txc.wg_note_encap(lib.make_batch(buf, n * slot, n, lib.MEM_DEVICE, stride=slot, length=length, peer=d(peer.view(np.int32))),
                              1420, t0 + k, wl)
            txc.sync()
            assert (wl == 80).all()
            wires.append(buf.cpu().numpy().reshape(n, slot))
            assert np.array_equal(wires[-1][:, 8:16].copy().view("<u8").reshape(-1), want)
            inner.append(rows[:, 16:16 + length].copy())
            ctrs.append(want)
            assert txc.filter_flows() == sent.flows()
        assert np.array_equal(txc.wg_send_counters(n_peers), nxt)
        # some of the flows are ours: what comes back on them passes whatever the rules say
        back = np.concatenate(inner)[::7].copy()
        back[:, 12:16], back[:, 16:20] = np.concatenate(inner)[::7, 16:20], np.concatenate(inner)[::7, 12:16]
        back[:, 20:22], back[:, 22:24] = np.concatenate(inner)[::7, 22:24], np.concatenate(inner)[::7, 20:22]
        flat = np.ascontiguousarray(back).reshape(-1)
        offs = np.arange(len(back), dtype=np.uint64) * length
        flows_in.note_outbound_batch(flat, offs, np.full(len(back), length, np.uint32), t0)
        rxc.filter_note_outbound(lib.make_batch(flat, flat.nbytes, len(back), lib.MEM_HOST, offsets=offs,
                                                lens=np.full(len(back), length, np.uint32)), t0)
        both, who, ctr, plain = np.concatenate(wires), np.concatenate([peer, peer]), np.concatenate(ctrs), np.concatenate(inner)
        filters = {}
        # the second half in order, then any of both again and again
        for k, pick in enumerate([np.arange(n, 2 * n), rng.integers(0, 2 * n, n), rng.integers(0, 2 * n, n)]):
            fresh = np.array([filters.setdefault(int(who[i]), O.ReplayFilter()).validate(int(ctr[i])) for i in pick])
            rows = both[pick].copy()
            want = np.full(n, lib.WG_REPLAY, np.uint8)
            got_in = np.flatnonzero(fresh)
            passed = flows_in.check_inbound_batch(np.ascontiguousarray(plain[pick[got_in]]).reshape(-1),
                                                  np.arange(got_in.size, dtype=np.uint64) * length,
                                                  np.full(got_in.size, length, np.uint32), t0 + 5 + k)
            want[got_in] = np.where(passed != 0, lib.WG_OK, lib.WG_FILTERED)
            wire, out = d(rows.reshape(-1)), torch.zeros(n * slot, dtype=torch.uint8, device="cuda:0")
            res, olen, gp = torch.full((n,), 99, dtype=torch.uint8, device="cuda:0"), i32(), i32()
            gc = torch.zeros(n, dtype=torch.int64, device="cuda:0")
            torch.cuda.synchronize()
            rxc.wg_decap_filter(lib.make_batch(wire, n * slot, n, lib.MEM_DEVICE, stride=slot, length=80),
                                lib.make_batch(out, n * slot, n, lib.MEM_DEVICE, stride=slot), t0 + 5 + k, res, olen, gp, gc)
            rxc.sync()
            assert np.array_equal(gc.cpu().numpy().view(np.uint64), ctr[pick])
            assert np.array_equal(res.cpu().numpy(), want)
            assert len(np.unique(want)) >= 2
            assert rxc.filter_flows() == flows_in.flows()


@pytest.mark.parametrize("n_peers,n", [(1, 257), (255, 300), (3, 1023), (254, 1024), (256, 700), (40, 2049), (255, 4096)])
def test_counters_and_windows_by_rows_of_a_workgroup(n_peers, n):
    """One row of 64 packets a wave and as many as four, the last ones part full, as few peers as one
    and as many as fit, and one more (which are sorted): the checks are those of the test above."""
    test_counters_and_windows_of_one_workgroup_over_the_peers_digits(n_peers, n)


@pytest.mark.parametrize("n_peers,n", [(1, 257), (255, 1025), (256, 1024), (40, 2048), (40, 2049), (255, 2047), (1024, 2048)])
def test_tunnel_batches_of_a_wave_per_packet_in_three_launches(n_peers, n):
    """The fewest and the most packets that are encapsulated in one launch and decapsulated in two, one
    more, as many peers as the second of those takes and more: the checks are those of the test of
    larger batches above."""
    test_tunnel_batches_whose_tiles_add_up_the_rows_before_theirs(n_peers, n)
