"""The workspace query for calls that the register-dequantising matmul takes (host only)."""


def test_query_has_room_for_the_split(cabi):
    """Few rows of a long K: staged rows and the partial sums of K split in four, where the
    decode launches' own split would hold the rows but not the partials."""
    for v, x, m, staged in ((cabi.CMK_IQ2_XS, cabi.CMK_BF16, 8, True),
                            (cabi.CMK_IQ2_S, cabi.CMK_BF16, 5, True),
                            (cabi.CMK_IQ3_S, cabi.CMK_BF16, 12, True),
                            (cabi.CMK_IQ2_XS, cabi.CMK_F16, 2, False),
                            (cabi.CMK_IQ2_XXS, cabi.CMK_BF16, 16, True)):
        align = lambda n: (n + 255) // 256 * 256  # noqa: E731
        # scales of the rows and of their 56 super-blocks, the rows
        rows = align(4 * m) + align(4 * 56 * m) + align(2 * 14336 * m) if staged else 0
        assert cabi.workspace_size(x, m, 4096, 14336, variant=v) == rows + 4 * m * 4096 * 4


def test_query_counts_row_pairs_past_2_31(cabi):
    """f32 rows are staged as pairs, 2^32 and more of them from 2^31 rows on."""
    def query(m):
        return cabi.workspace_size(cabi.CMK_F32, m, 2, 8, variant=cabi.CMK_IQ2_XS)
    assert query((1 << 31) + 64) >= query((1 << 31) - 64)


def test_query_is_bounded(cabi):
    """Staged rows of one pass (256 MB and their scales), not of all rows; and nothing more
    than the decode launches' split where the matmul cannot run: rows too long for its 32-bit
    offsets, 2 GB of weights and more."""
    mb = 1 << 20
    align = lambda n: (n + 255) // 256 * 256  # noqa: E731
    for x in (cabi.CMK_F32, cabi.CMK_BF16):
        rows = 256 * mb // (28672 * (4 if x == cabi.CMK_F32 else 2)) // 128 * 128
        bytes_ = rows * 28672 * (4 if x == cabi.CMK_F32 else 2)
        got = cabi.workspace_size(x, 65536, 28672, 28672, variant=cabi.CMK_IQ2_XS)
        assert bytes_ < got <= 256 * mb + align(4 * rows) + align(4 * 112 * rows)
    assert cabi.workspace_size(cabi.CMK_F32, 200, 1, 8 * mb, variant=cabi.CMK_IQ2_XS) <= 4 * mb
    assert cabi.workspace_size(cabi.CMK_F32, 200, 1 << 18, 32768, variant=cabi.CMK_IQ2_XS) <= 4 * mb
