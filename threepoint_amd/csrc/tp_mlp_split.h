// tp_mlp_split.h -- how a training batch is split for the weight-gradient product (k_gemm_wgrad, tp_mlp.hip).
// Plain C++, so that the bound the workspace relies on is checked on the CPU for every batch size.
#pragma once

struct TpWgradSplit {
    int rows;  // rows per split, a multiple of 32 (the last split may be shorter)
    int n;     // splits; each holds at least one row
};

// The most splits a batch of up to `rows` rows takes: one per 256 rows, up to 64.  Never falls as rows grows, so a
// workspace sized for its capacity serves every smaller batch.
constexpr int tp_wgrad_max_splits(int rows)
{
    return rows < 512 ? 1 : rows >= 64 * 256 ? 64 : rows / 256;
}

// The split of a batch of M >= 1 rows, from M alone: a batch's gradient has the same bits whatever batches came before it.
// The quotient is rounded up before it is rounded to 32, so that n rows-sized splits cover M with n <= the bound above.
constexpr TpWgradSplit tp_wgrad_split(int M)
{
    const int want = tp_wgrad_max_splits(M), per = M / want + (M % want != 0);
    const int rows = per / 32 * 32 + (per % 32 != 0 ? 32 : 0);
    return TpWgradSplit{rows, M / rows + (M % rows != 0)};
}
