"""The numbers by which the dispatcher chooses between kernels that compute the same thing.

They were measured on one MI355X with the layer sizes of the Llama-3-8B shape (and checked on
the Llama-2-7B and Llama-3-70B shapes): they change which kernel runs and how it is launched,
never what comes out, so another shape or another card may want other numbers and nothing
else.  All of them are here, as data; ``ops`` and ``parts.linear`` read ``TUNING`` and hold
no such number of their own.  Replace fields (``dataclasses.replace``) or assign ``ops.TUNING``
to try others.
"""
from __future__ import annotations

from dataclasses import dataclass


@dataclass(frozen=True)
class Tuning:
    # ---- the weight-streaming product for few rows (gemm_skinny.hip)
    skinny_rows: int = 16               # up to here it beats the library's product with a plain weight ...
    skinny_rows_packed: int = 24        # ... up to here with a packed weight, whose epilogues save the kernels around it
                                        # (whole decode steps: +9 % at 17 rows, +4 % at 24)
    skinny_rows_short_k: int = 24       # ... and up to here for packed weights with K <= skinny_short_k (q/k/v, output,
                                        # gate/up; it was 32 before the row-sharing product spread its tiles over all compute
                                        # units: now whole steps of 28 requests are 1 % faster and of 32 requests 2.7 % with 24)
    skinny_short_k: int = 8192
    skinny_rows_any_weight: int = 4     # so few rows always go to it
    skinny_small_weight: int = 1 << 24  # without a packed copy, beyond 4 rows only weights up to this many elements
    skinny_two_tiles_from: int = 6144   # packed: two tiles of 16 features a workgroup from this many features on ...
    skinny_four_tiles_from: int = 65536  # ... four for the widest, with more than 8 rows
    skinny_workgroups_per_cu: int = 4   # plain: as many tiles as still leave this many workgroups for each compute unit
    skinny_eight_waves_to: int = 8192   # eight waves share a workgroup's K up to this many output features, four beyond
    compute_units: int = 256            # of the card the numbers were measured on; ``for_device`` puts in the card's own
    # ---- the product that shares the rows through LDS (gemm_mid.hip, up to 256 rows)
    mid_long_k: int = 8192              # with a plain (not packed) weight only weights with a longer K than this (the down
                                        # projection) go to it at all; a packed weight with a longer K goes to it
    mid_long_k_rows: int = 11           # ... above this many rows (whole decode steps: 0.9 % faster at 12 rows, 3 % at 16;
                                        # 0.3 % slower at 11: below, the weight-streaming kernel with the norm in its epilogue)
    mid_swiglu_features: int = 8192     # gate/up with SwiGLU goes to it from this many rows of the weight on,
    mid_swiglu_rows: int = 14           # above this many rows of the batch (whole steps: 2.8 % at 16 rows, nothing at 14, slower below)
    mid_swiglu_max_rows: int = 192      # ... up to this many (at 160 and 192 rows 57 and 61 us against the library's 62 and 66 with
                                        # the activation kernel: whole steps 4 and 6 % faster; at 256 rows 78 against 73)
    mid_long_k_max_rows: int = 256      # the products cut over K go to it up to this many rows with a long K (the down
                                        # projection: 31 us at 121 rows, 42 against the library's 85 at 160, 55 against 65 at 256)
    mid_short_k_max_rows: int = 192     # ... and up to this many with a shorter one (the output projection: 19 us against 25 to
                                        # 28 at 160 to 192 rows, no gain beyond)
    mid_qkv_rows: int = 16              # q/k/v with the rotation and the cache write in its epilogue goes to it above this
    mid_qkv_max_rows: int = 192         # many rows and up to this many, with a packed weight (whole decode steps over short
                                        # contexts: 1 to 2 % faster from 20 to 64 rows, 2.5 % at 80, 3.5 % at 128, 5 % at 144, even at 160
                                        # to 192; 1 to 2 % slower at 14 and 16 rows)
    mid_qkv_one_round_rows: int = 32    # ... beyond this many rows only if its workgroups (one for every 32 rows of the weight) are
                                        # no more than the compute units
    mid_add_norm_rows: int = 16         # a product with a short K that ends a branch (the output projection) goes to it with the residual
    mid_add_norm_max_rows: int = 32     # sum and the next norm's weight in its epilogue above this many rows and up to this many, while
                                        # its workgroups (one for 16 output features) run in one round: 11.9 us at 17 to 32 rows (the
                                        # weight-streaming kernel 13.1 to 16.9, planes and the norm kernel 14.2); whole steps 0.3 %
                                        # faster at 20 rows, 1.7 % at 32; 2 % slower at 16 and at 40 to 48, where the first product
                                        # of the feed-forward pays more for the rows' factors than the norm kernel cost
    mid_f32_rows: int = 32              # a product with 32-bit output (the output matrix, 1.05 GB) goes to it, uncut, above this many
    mid_f32_max_rows: int = 64          # rows and up to this many (193 / 195 us against the library's 215 / 219 at 48 / 64 rows; whole steps at 25 to 32 rows: nothing) ...
    mid_f32_wide_max_rows: int = 128    # ... and where its workgroups of 256 features fill their rounds (mid_ring_wide in gemm_mid.hip) up to so many (198 and 202 us
                                        # against 235 and 246 at 96 and 121 rows)
    mid_min_slice_steps: int = 4        # a slice of K keeps at least this many macro-steps of 128
    mid_max_slices: int = 8
    # ---- the product whose waves share out K (gemm_wavek.hip, up to 64 rows)
    # (its numbers stand in gemm_wavek.hip; measured with 64 to 8192 features, K of 128 to 4096 and the matrix out of memory)
    wavek_wide_per_cu: int = 16         # 32 features a workgroup instead of 16 beyond so many features a compute unit (4096 x 2048 at 4 / 33 rows: 6.2 / 9.8 us
                                        # with 32, 5.4 / 8.4 with 16; 5120 x 2048 6.4 / 9.9 and 7.0 / 14.8)
    wavek_max_k: int = 4096             # the longest K measured (4096 features, K = 4096: 8.6 us against the weight-streaming kernel's 9.1 at 16 rows, 10.7
                                        # against 14.4 and the library's 13.2 at 32, 14.7 against 15.3 at 64)
    wavek_short_k: int = 1024           # with a K below it is the fastest at any number of rows (2048 x 512: 2.7 us against 2.8 at 1 row, 3.4 against 3.8 at 24, 4.2
                                        # against the library's 7.0 at 64; 16 groups of 128 x 128 2.5 against 2.8 at 8 rows, 2.8 against 4.6 at 32, 3.2 against 4.9 at 64)
    wavek_few_rows: int = 8             # up to here a plain product goes to it beyond wavek_wide_per_cu only (5120 x 2048: 6.4 us against 6.8 at 8 rows; with 2048
                                        # features 4.4 and 4.4); from 9 rows on 0.97 of the weight-streaming kernel's time, at 24 0.92
    wavek_wide_few_rows: int = 12       # ... up to here beyond wavek_wide_few_features with a K up to wavek_wide_few_k (4096 x 1408 at 9 and 12 rows 5.0 and 5.0 us
    wavek_wide_few_features: int = 3072  # against the weight-streaming kernel's 4.7 and 4.7, 4096 x 2816 7.1 and 6.9 against 6.9 and 6.7; 3072 x 2048 5.3 and 5.3, 4096 x 4096
    wavek_wide_few_k: int = 2816        # 9.0 against 9.1)
    wavek_few_group_rows: int = 4       # ... up to here a product in groups (2 of 1024 x 1024 with a gate at 8 rows: 4.0 us against 4.4; without one 3.4 to 3.5 either way)
    wavek_two_tiles_k: int = 3840       # with a longer K, and features from skinny_two_tiles_from on, the weight-streaming kernel is faster up to
    wavek_two_tiles_rows: int = 16      # so many rows (8192 x 4096: 15.0 us against 13.5 at 1 to 16 rows, 16.8 against 16.7 at 17; 6144 x 4096 11.8 to 12.5 against 11.3 to 12.0;
                                        # 8192 x 3840 12.4 to 13.3 against 12.8 to 13.5)
    wavek_few_features: int = 1024      # few workgroups, each with much to do: below so many features not where K times the rows is beyond
    wavek_few_features_work: int = 98304    # this (512 x 4096 at 64 rows 12.6 us against the library's 11.3, 64 x 2048 7.5 against 5.2; at 48 6.4 against 7.7)
    wavek_least_features: int = 64      # below so many, and a K that is not short, only up to
    wavek_least_rows: int = 24          # so many rows (16 x 1024: 3.6 us against 3.9 at 24, 4.2 against 3.9 at 48)
    wavek_many_features: int = 6144     # beyond so many features, with a K beyond wavek_short_k, up to
    wavek_many_rows: int = 48           # so many rows (8192 x 2048 at 64 rows 12.4 us against the library's 13.7 with the matrix out of memory, 11.8 against 11.0 in a
                                        # model that runs its layers in a loop and finds it in the last-level cache; 10.7 against 13.9 at 48)
    wavek_library_rows: int = 48        # above so many rows and below 64, up to wavek_library_features and with a K beyond wavek_library_k, the library's plain product is
    wavek_library_features: int = 4096  # faster (2048 x 3072: 11.1 us against 10.3 at 49 to 63 rows, 11.1 against 15.6 at 64, 10.0 against 10.3 at 48; 4096 x 4096 15.0 against
    wavek_library_k: int = 2688         # 14.0; 1280 x 2816 9.9 against 9.6; 1024 x 2816 9.7 against 11.2, 2048 x 2688 9.7 against 13.6, 4352 x 4096 15.9 against 16.9)
    wavek_swiglu_least: int = 512       # gate and up rows and K from which on SwiGLU was measured (1024 x 512 to 8192 x 4096: the library's product alone, without
                                        # the activation kernel's 2 us, is 1 us faster at most, at 48 rows of 2816 x 3072; the row-sharing kernel 1.5 us slower at 64 rows and 0.9
                                        # faster at 24 to 32 rows of 8192, which go to it: mid_swiglu_features).  With that kernel, matrices out of memory, at 33, 48, 49 and 63 rows: 2048 x 3072 11.3,
                                        # 11.5, 12.4, 12.5 us against the library's 12.7, 12.6, 12.6, 12.8, 1536 x 4096 13.1, 13.4, 14.6, 15.1 against 14.5 (out of the last-level cache the
                                        # library's are 10.2 and 11.4)
    wavek_qkv_rows: int = 32            # q/k/v with the rotation and the cache write in its epilogue goes to it above so many rows and up to 64, where the row-sharing
                                        # kernel would be taken, whatever K (us at 33, 48 and 64 rows, 48 heads of 128, K = 4096: 17.8, 18.3, 19.5 against 19.0, 19.2, 21.2, K = 8192:
                                        # 28.2, 30.2, 32.0 against 32.6, 31.0, 35.1; 24 heads, K = 512: 6.1, 6.4, 7.2 against 6.2, 6.3, 7.5, K = 2048: 10.5, 10.9, 12.3
                                        # against 10.7, 10.5, 12.6; 8 heads of 64, K = 8192: 21.8, 23.4, 26.6 against 27.8, 27.8, 31.2; measured for 8 to 64 heads); 15.5
                                        # against 14.8 at 24 rows, 48 heads, K = 4096
    # ---- the product of many rows in tiles (gemm_tiles.hip), us of the library's and of it
    tiles_rows: int = 256               # above so many rows (fewer have kernels of their own)
    tiles_swiglu_k: int = 2048          # SwiGLU with a longer K stays with the library (28672 x 4096: 83 and 95 at 300 rows, 290 and 306 at 1,500; 5632 x 2048 51.8 and 49.3
                                        # there, 59.7 and 52.4 at 2,014; 2816 x 1024 26.3 and 18.8)
    tiles_library_tile: int = 96        # with a K from tiles_library_k on the library's tiles of 96 x 128, where they fill a round to seven eighths or more, are faster than one of
    tiles_library_k: int = 4096         # 128 x 128 that is less full (4096 x 4096 at 640 / 700 / 765 rows 36.5 / 32.6 / 34.1 and 37.8 / 33.2 / 38.2; 4096 x 14336 112 / 100 / 106 and 130 / 113 / 129;
                                        # 5120 x 4096 at 512 and 576 36.5 / 32.9 and 38.1 / 33.5), below and beyond not (4096 x 4096 at 576 / 800 36.6 / 39.8 and 33.5 / 31.7, 5120 x 4096 at 450 / 640 35.1 / 39.6 and
                                        # 33.1 / 38.1), and with a shorter K neither (3072 x 2048 at 765 19.4 and 15.9, 2048 x 2816 at 1,280 22.6 and 20.6, at 1,400 21.1 and 21.7)
    tiles_short_k: int = 2048           # a round of 128 x 256 up to five eighths full only with a K up to this (4096 x 2048, 1,100 rows: 27.0 and 24.3; 2560 x 2048, 2,014: 27.8 and
                                        # 25.0; 4096 x 4096, 1,100: 42.6 and 42.8), and with this K not one less than three fifths full (3072 x 2048 at 1,400 23.6 and 24.7, 5632 x 2048 at 661 23.3 and 25.9)
                                        # (a fuller round, with any K, is no gain in a whole prompt, where the card's power limit lets every kernel pay for another's work: 4096 x
                                        # 14336, 2,048 rows, 210 and 196 alone, 225 and 204 inside an 8-layer prompt of the 8B shape, which takes 6.79 and 6.85 ms)
    tiles_any_k: int = 1024             # with a longer K a round that the rows and features that are there fill to less than half (SwiGLU: two fifths) is the library's: 6144 x 2048 at 300 rows 15.5 and 16.2 (32-bit
                                        # sums 16.0 and 19.4), 3584 x 3584 at 513 / 576 / 640 23.1 / 23.0 / 26.0 and 25.1 / 25.0 / 24.0; 2816 x 1024 at 700 11.6 and 11.0.  SwiGLU in tiles of 256 x 256 from this K on has
                                        # to fill more than two and a half rounds of square tiles: 11264 x 2048 at 576 / 800 / 1,000 36.3 / 43.0 / 58 and 44.9 / 46.3 / 49, 5632 x 2048 at 1,400 / 2,014 39.6 / 59.7 and 48.8 / 50
    tiles_tall_k: int = 2048            # a longer K with half as many rows again as features is the library's (768 x 3072 at 3,471 22.9 and 25.6, 1024 x 2816 at 2,841 22.9 and 24.2; 960 x 1536 at 3,552 1.08 times as fast
                                        # in tiles), with any K once a round is nine tenths full and a fifth more rows than features (1536 x 1536 at 2,300 / 2,547 rows 1.09 and 0.82 times as fast, 1792 x 3072 at 2,249 0.86)
    tiles_long_k: int = 4096            # a longer one with nine tenths as many rows as features (2048 x 8192 at 2,048 66.8 and 70.5, 1024 x 8192 at 4,000 68.1 and 78.5), or a round less than five eighths full, or so full with a third as many rows as features (2048 x 14336
                                        # at 1,117 107 and 121, 2944 x 5632 at 688 34.2 and 37.4, 2560 x 11008 at 1,004 86 and 93; 4096 x 14336 at 513 1.14 times as fast in tiles)
    # ---- the library's product of many rows (parts/linear.library_friendly_rows)
    library_rows: int = -1              # rows of zeros behind each half of a plain gate/up matrix: -1 times the library once per
                                        # shape at load and fills up where that is 15 % faster (the outcome can differ from box
                                        # to box near that mark); 0 never fills up; n > 0 fills each half up to a multiple of n
    # ---- the decode attention's cut of a request's keys into parts (attention_mfma.hip)
    decode_min_part_keys: int = 512     # a part of so many keys; up to 512 keys one part (the longest context rounded up to a power of two).  One MI355X, us, 16 heads over 4, 1 / 2 / 4 / 8
                                        # parts with their second kernel: 4 requests of 500 keys 6.6, 7.8, 6.8, 6.7, 8 of 300 6.6, 7.7, -, 7.1, of 500 8.7, 8.9, 7.7, 7.3 (the one case in which parts gain)
    decode_max_parts: int = 32
    decode_few_parts: int = 8           # beyond 512 keys up to so many parts, however short (of at least 64 keys: 513 are taken for 1,024).  4 requests of 1,000 keys 12.6, 10.9, 8.9, 7.5,
                                        # 8 of 1,000 13.8, 11.6, 9.3, 8.3, 1 of 2,000 18.6, 11.1, 9.2, 7.7
    decode_long_keys: int = 1024        # beyond so many keys of the longest request eight waves a workgroup for one to two workgroups a compute unit (attention_mfma.hip).  Lengths of 10 to 100 % and of 50
                                        # to 100 % of it, 8 waves' time over 4's: 512 workgroups of heads of 128 at 500 / 1,000 / 1,500 / 3,000 keys 1.05 / 0.98 / 0.95 / 0.96 and 1.08 / 1.01 / 1.00 / 0.95, 384 of heads of
                                        # 64 1.10 / 0.99 / 0.83 / 0.82 and 1.21 / 1.06 / 1.01 / 0.95; 768 and more 1.02 to 1.14 from 1,000 to 1,500 keys on
    decode_long_part: int = 768         # from so many keys a part on four waves for parts of heads of 128 that fill more than half of the chip: eight parts of 32 to 256 workgroups, 8 waves' time over 4's at 250 / 500 /
                                        # 1,000 / 2,000 keys a part 0.93 to 1.01, 0.93 to 1.01, 1.01 to 1.07, 1.02 to 1.05
    decode_few_workgroups: int = 128    # up to this many workgroups without parts: about one workgroup per compute unit
    decode_long_context: int = 2048     # between half the chip's worth of workgroups and all of it: parts only from here on
                                        # (rounded up to a power of two: from 1,025 keys),
    decode_long_part_keys: int = 1024   # of at least this many keys (with non-temporal loads of the keys, whole decode steps over
                                        # 2k keys: 5.5 % faster at 17 requests, 3.5 % at 20, 1.7 % at 22, nothing from 24 on),
    decode_long_max_parts: int = 4      # at most this many,
    decode_fill_slack: float = 0.07     # the fewest that fill whole waves of workgroups within this of the best


TUNING = Tuning()


def for_device(tuning: Tuning, device) -> Tuning:
    """``tuning`` with the facts of the card at ``device`` in the fields that are the card's (the number of compute
    units), not choices."""
    import dataclasses

    import torch
    units = int(torch.cuda.get_device_properties(device).multi_processor_count)
    return tuning if units == tuning.compute_units or units <= 0 else dataclasses.replace(tuning, compute_units=units)
