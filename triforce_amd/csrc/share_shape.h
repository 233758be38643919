// How the one-workgroup-per-CU products (share_gemm.h, gemv_wide.hip) deal `panels` 16-row weight panels to 256 workgroups.
#pragma once

// `each` whole panels a workgroup, and `rest` (0, 4, 8 or 12) of the `left` rows that are left over.  each == 0: not a shape of these forms.
struct ShareShape { int each, left, rest; };

// pairs: panels of 8 gate | 8 up rows, whose rows are dealt in pairs; whole_rows: rows that have to come in whole panels; rows: of the operand.
static inline ShareShape share_shape(int panels, bool pairs, int whole_rows, int rows) {
    const int whole = panels / 256, left = (panels - 256 * whole) * 16, per = (left + 1023) / 1024 * 4;
    if (panels < 256) return {0, 0, 0};
    if (per > 0 && per < 16 && 256 * whole * 16 < whole_rows) return {0, 0, 0};
    // One panel and a rest of up to 4 rows, from the third (gate | up) or fifth row block on: every block reads the rest again at the price of a
    // panel.  300 panels, K 4 096, gate | up, 64 / 128 / 256 rows here 26.5 / 48.6 / 92.9 us, panel by panel 25.1 / 39.9 / 76.4; other outputs
    // 23.5 / 44.5 / 86.8 and 25.6 / 41.8 / 80.8
    if (whole == 1 && per == 4 && rows > (pairs ? 32 : 64)) return {0, 0, 0};
    // Rests of 9 to 12 rows a workgroup, and of 5 to 8 beside one panel of gate | up, cost as much as a panel of their own or more (gate | up deals
    // them in pairs of rows, 32 bytes each): whole panels on fewer CUs.  us at one row, K 4 096, gate | up: 448 panels 13.0 panel by panel, 16.3
    // with a rest, 12.9 on 224 CUs; 688 17.8, 21.9, 16.7; other outputs 448 12.5, 12.7, 12.5; 688 17.0, 18.3, 16.1; 900 21.7, 21.3 and, as 1 024,
    // 22.7.
    const bool up = per == 16 || (per == 12 && (pairs || whole <= 2)) || (per == 8 && pairs && whole == 1);
    if (per == 0 || up) return whole + up > 8 ? ShareShape{0, 0, 0} : ShareShape{whole + up, 0, 0};
    return whole > 7 ? ShareShape{0, 0, 0} : ShareShape{whole, left, per};
}
