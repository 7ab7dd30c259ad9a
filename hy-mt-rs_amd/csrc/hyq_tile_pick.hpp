// The tile shape of a batched product (the shapes: hyq_gemm.hip). Host code only.
#pragma once

namespace hyq {

enum TileShape { T256, T256R96, T192, T128, T64 };

// The tile shape of a dense product: the one whose workgroups take the least
// time in rounds over the 256 CUs. rows(r): row tiles of r rows. A shape's
// time is that of a 64-column step with one workgroup on a CU (us, Q4_K
// [14336 x 4096]: 67 us for 64 steps of 224 workgroups of 256 tokens), `pair`
// with two (Tile128, Tile64). All shapes give an element the same bits, so the
// choice is free. By 256, 192, 128 tokens and 64 rows x 256 tokens: Q2_0C
// [12288 x 2048] at 777 tokens 71 / 67 / 71 / 63 us, Q4_K [14336 x 4096] at
// 130 tokens 57 / 52 / 47 / 40 us, 384: 71 / 66 / 78 / 76, 512: 77 / 109 / 88
// / 83, 777: 130 / 147 / 142 / 136.
template <class Rows>
inline TileShape pick_tile(int batch, int kslices, bool r96, const Rows &rows)
{
    struct Shape {
        TileShape s;
        int rows, tokens;
        float time, pair;
    };
    static constexpr Shape shapes[] = {{T256, 128, 256, 1.06f, 0.f},
                                       {T256R96, 96, 256, 0.85f, 0.f},
                                       {T192, 128, 192, 0.9f, 0.f},
                                       {T128, 128, 128, 0.73f, 1.25f},
                                       {T64, 64, 256, 0.5f, 1.08f}};
    TileShape best = T256;
    float least = 1e30f;
    for (const Shape &c : shapes) {
        if (c.s == T256R96 && !r96) continue;
        const long wgs = (long)rows(c.rows) * ((batch + c.tokens - 1) / c.tokens) * kslices;
        const long full = c.pair ? wgs / 512 : wgs / 256, rest = c.pair ? wgs % 512 : wgs % 256;
        const float time = (float)full * (c.pair ? c.pair : c.time) +
                           (rest == 0 ? 0.f : rest <= 256 ? c.time : c.pair);
        if (time < least) {
            least = time;
            best = c.s;
        }
    }
    return best;
}

// Row tiles of r rows of a weight of M rows, and of a gate/up product of 2 x
// M rows (a tile holds r / 2 of each).
inline int matmul_row_tiles(int M, int r) { return (M + r - 1) / r; }
inline int gate_up_row_tiles(int M, int r) { return (M + r / 2 - 1) / (r / 2); }

} // namespace hyq
