// Which products gemm256_kernel takes (gemm.hip), a plain function of the shape and of the number of compute units.
#pragma once
#include <cstdint>
#include <initializer_list>

// GELU_CACHED: as GELU, the outputs left to the caches; GELU_ONLY: the activation alone
enum EpilogueMode { EPI_PLAIN = 0, EPI_RESIDUAL = 1, EPI_GELU = 2, EPI_GELU_BWD = 3, EPI_GELU_CACHED = 4, EPI_GELU_ONLY = 5 };

// Which products the 256-row kernel takes, and with which width: the least of estimated costs in columns times k.  Each of
// a unit's rounds of tiles costs, per k, its width and a share that does not depend on it, and an epilogue by outputs; the
// 128-row blocks, two to a unit, cost the same by pairs, where a lone block takes more than half a pair's time.  Of 128 and 192 columns the
// cheaper counts there: priced at 192 alone, GELU' took half a round of 256-row tiles where two blocks of 128 fit every unit (3584 x 1920, K = 1024
// 26.3 us, 20.8; 4352 x 3456, 2816 109, 90).  The constants are a fit to products of 2048 to 16384 rows at the widths of models of 256 to 1024
// columns, plain, residual and with either GELU: over 1512 of them, of 1920 to 16384 rows, the choice is within 0.5 % of the best of the four
// (geometric mean), where taking 192 or else 128 columns for tiles that fill 90 % of the last round was within 2.7 %; over 7140 at any
// width from 256 to 4096 within 1.7 %, and slower than 128-row blocks by more than 3 % at 25 of them, by 11 % at worst.  Products of less than
// 768 of k (512 with a GELU) don't pay for a lone block's cold start, nor do 128 columns of less than 768, or with GELU', unless
// they fill the units and 192 does not divide the width (2176 x 3584 x 896 21.3 us on 128-row blocks, 23.0 on 128 columns).
// The forward GELU of widths that 192 divides stays with the 128 x 192 blocks: alone they are as fast (16384 x 3072 x 768 99.0 us,
// with 256 columns 97.9), but inside a step the second block covers the writes of two results (eight steps at d_model 768 183.0 ms,
// with 256 columns 187.1).  Rows that 128 divides and 256 does not: the half tiles count as whole ones, and over the same products of
// 4224 to 16256 rows the choice takes 1.5 to 6.1 % less than 128-row blocks alone (10368 x 1024 x 4096 100.3 -> 79.2 us,
// 16256 x 768 x 3072 75.6 -> 59.8), at 2176 rows 0.2 %.
inline int columns_of_256(int M, int N, int K, int mode, int units) { // 0: the 128-row blocks
    const bool gelu = mode != EPI_PLAIN && mode != EPI_RESIDUAL;
    const int wide = N % 192 == 0 ? 192 : 128;
    const int64_t blocks = int64_t(M / 128) * (N / wide), per_unit = (blocks + units - 1) / units;
    if (M % 128 || K % 128 || per_unit < 2 || K < (gelu ? 512 : 768))
        return 0;
    if (gelu && mode != EPI_GELU_BWD && wide == 192)
        return 0;
    double best = 0;
    for (int width : {128, 192}) { // both, as the blocks of either may be the ones taken
        if (N % width)
            continue;
        const int64_t on_unit = (int64_t(M / 128) * (N / width) + units - 1) / units;
        const double cost = (double(on_unit / 2) + on_unit % 2 * 0.83) * (double(K) * (width + (gelu ? 100 : 86)) + width * (gelu ? 810. : 410.));
        if (best == 0 || cost < best)
            best = cost;
    }
    int columns = 0;
    for (int bn : {128, 192, 256}) {
        if (N % bn)
            continue;
        const int64_t tiles = int64_t((M + 255) / 256) * (N / bn), rounds = (tiles + units - 1) / units;
        if (bn == 128 && (K < 768 || mode == EPI_GELU_BWD) && (wide == 192 || tiles * 10 < rounds * units * 9))
            continue;
        const double cost = double(rounds) * (double(K) * (bn + 52) + bn * (gelu ? 1050. : 480.));
        if (cost < best)
            best = cost, columns = bn;
    }
    return columns;
}
