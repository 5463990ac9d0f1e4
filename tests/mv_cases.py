"""Plans of the exact MULTISEQ kernel (kq_mv.hip) that between them run every
form of it: rows of at most 128 chunks (H = 1: 8 waves, 8 rows a task) and
longer ones (H = 2: 16 waves, 2 rows), S = 2, 3, 4 streams a group, no full
turn of tasks or one, and a last turn whole or cut into pieces of 1 or 2
streams."""

SHAPES = {1: (8, 8), 2: (16, 2)}        # H: waves, rows of a task
ROWS = {1: 1280, 2: 8448}               # H: a tile of chunks and a remainder


def cut_of(S, rem, W):
    """Pieces of a left-over task (mv_cut): one a wave."""
    return S if S * rem <= W else 2 if S == 4 and 2 * rem <= W else 1


def form(H, S, ng, mc):
    """(full turns, tasks left over, their pieces) of an item."""
    W = SHAPES[H][0]
    full, rem = divmod(ng * -(-mc // S), W)
    return full, rem, cut_of(S, rem, W) if rem else 0


def plans():
    """(H, S, row groups per item, streams per chunk, streams) of each."""
    out = []
    for H, (W, _) in SHAPES.items():
        for S in (2, 3, 4):
            for full in (0, 1):
                # left over: none, one, half the waves, one more, all but one
                for rem in (0, 1, W // 2, W // 2 + 1, W - 1):
                    if full or rem:
                        out.append((H, S, full * W + rem, S, S))
            # two and more groups of streams, a short last group and chunk
            out += [(H, S, 2, 8, 8), (H, S, 3, 7, 13), (H, S, 5, S + 1, 3 * S + 2), (H, S, 1, 8, 17)]
    return out
