"""Which form of the workgroup attention kernel a step's prompt portions go to."""
from kv_cache_optimization_for_llm_amd.ops import attention as A


def test_lines_between_the_forms():
    kind = A.choose_lds_kind
    for groups, mean, dim, by_workgroup, want in (
            (512, 1024.5, 64, False, A.LDS_TWO_GROUPS), (447, 1024.5, 64, False, A.LDS_BLOCKS_OF_32), (632, 660, 64, False, A.LDS_BLOCKS_OF_32),
            (699, 1100, 64, True, A.LDS_TWO_GROUPS), (699, 2048, 64, True, A.LDS_BLOCKS_OF_32), (700, 1100, 64, True, A.LDS_BLOCKS_OF_64),
            (2048, 4095, 64, True, A.LDS_BLOCKS_OF_64), (896, 100, 64, True, A.LDS_BLOCKS_OF_32), (1024, 512, 64, True, A.LDS_BLOCKS_OF_64),
            (1025, 2800, 64, True, A.LDS_BLOCKS_OF_32), (1025, 4096, 64, True, A.LDS_BLOCKS_OF_64), (1300, 1024, 64, True, A.LDS_BLOCKS_OF_64),
            (700, 1100, 64, False, A.LDS_BLOCKS_OF_32), (271, 1024, 128, False, A.LDS_BLOCKS_OF_32), (272, 512, 128, False, A.LDS_TWO_GROUPS),
            (272, 511, 128, False, A.LDS_BLOCKS_OF_32), (544, 2047, 128, True, A.LDS_TWO_GROUPS), (544, 4096, 128, True, A.LDS_BLOCKS_OF_32),
            (576, 1152, 128, True, A.LDS_BLOCKS_OF_64), (632, 656, 128, True, A.LDS_BLOCKS_OF_64), (768, 656, 128, True, A.LDS_BLOCKS_OF_32),
            (768, 4500, 128, True, A.LDS_BLOCKS_OF_32), (900, 1800, 128, True, A.LDS_BLOCKS_OF_32), (1100, 2800, 128, True, A.LDS_BLOCKS_OF_32),
            (1536, 4095, 128, True, A.LDS_BLOCKS_OF_32)):
        assert kind(groups, mean, dim, by_workgroup) == want, (groups, mean, dim, by_workgroup)
    # every line over mean keys is one at which captured steps are told apart
    lines = [entry for rule in (A._TWO_GROUPS, A._LONG_BLOCKS) for entries in rule.values() for entry in entries]
    assert {line for entry in lines for line in entry[2:]} <= set(A.MEAN_KEYS_STEPS) | {1 << 30}


def test_portions_keep_the_kernels_that_are_faster_for_them():
    """(lengths, mean keys, query heads a key head, head size) -> (wavefronts an item, 0 or one more than the form), each with the us that were measured
    for it and for the other form."""
    for lens, mean, group, dim, want in (
            ([2048], 1024.5, 4, 64, (1, 1 + A.LDS_TWO_GROUPS)),             # 34 / 39 by two wavefronts an item
            ([2047], 1024, 4, 64, (2, 0)),                                  # 44 in two groups / 42
            ([2600], 1300.5, 4, 64, (1, 1 + A.LDS_TWO_GROUPS)),             # 45 / 55 in blocks of 32
            ([319] * 6, 4168, 4, 64, (4, 0)),                               # behind 512 to 16,000 keys: 283 in two groups / 141
            ([905] * 2, 3581, 4, 64, (4, 0)),                               # behind 256 and 6,000: 126 / 93
            ([2173], 9279, 4, 128, (1, 1)),                                 # 443 / 428 in blocks of 32
            ([200] * 16, 100.5, 4, 64, (1, 1)),                             # 18 in blocks of 64 / 14
            ([1601, 676], 663, 4, 128, (1, 1 + A.LDS_TWO_GROUPS)),          # 52 / 62 in blocks of 64
            ([1248] * 2, 624.5, 4, 128, (1, 1 + A.LDS_BLOCKS_OF_64)),       # 42 / 53 in two groups
            ([1120] * 3, 560.5, 3, 128, (1, 1 + A.LDS_BLOCKS_OF_64)),       # 41 / 53, rows that end inside a workgroup but not inside a wavefront
            ([1000] * 3, 4500.5, 4, 128, (1, 1)),                           # 250 / 211
            ([5885], 7039, 3, 128, (1, 1)),                                 # 528 / 507
            ([3072], 1536.5, 4, 64, (1, 1 + A.LDS_BLOCKS_OF_64))):          # 59 / 66 in blocks of 32
        assert A.portion_choice(lens, mean, group, 8, dim, 16) == want, (lens, mean, group, dim)
