"""Which block of the GEMM a product takes on a part of 256 compute units (the rules of csrc/pq_gemm.hip and csrc/pq_tiles.h),
for tests that name the kernel their shapes are there for."""
CUS = 256


def _up(a, b):
    return -(-a // b)


def channel_block(M, N):
    """Packed operands, per-channel scales."""
    small, big = _up(M, 128) * _up(N, 128), _up(M, 256) * _up(N, 256)
    if _up(M, 32) * _up(N, 64) <= CUS:
        return "split K, 64 x 32"
    if _up(M, 64) * _up(N, 64) <= CUS:
        return "split K, 64 x 64"
    if _up(M, 128) * _up(N, 256) >= 1024 or (big <= CUS and small > 2 * CUS):
        return "256 x 256"
    if small > CUS and _up(M, 256) * _up(N, 128) <= CUS:
        return "128 x 256"
    return "128 x 64" if small < 128 else "128 x 128"


def group32_block(M, N):
    """Group-32 scales, no low-rank term."""
    blocks, halves = _up(M, 128) * _up(N, 128), _up(M, 64) * _up(N, 128)
    if _up(M, 32) * _up(N, 64) <= 5 * CUS:
        return "64 x 32"
    if blocks <= 2 * CUS or 10 * 2 * _up(blocks, CUS) > 11 * _up(halves, CUS):
        return "128 x 64"
    return "128 x 128"


def whole_tiles(tiles, K, wgx=CUS // 8):
    """Persistent products: lengths of an XCD's lists, shorter and longer (the same where tiles % 8 == 0), and of each the
    tiles that go out whole."""
    lengths = (tiles // 8, tiles // 8 + (1 if tiles % 8 else 0))
    past = max(n % wgx for n in lengths)
    rounds = tiles // 8 // wgx
    if K >= 4096:
        quarters = past <= wgx // 4
    else:
        quarters = rounds <= 4 and (past < wgx / 4 if K >= 2048 else past <= wgx / 6)
    return lengths, tuple(n - n % wgx if quarters else n for n in lengths)
