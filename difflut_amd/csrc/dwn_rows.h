// A DWN layer on few rows in one launch (dwn_rows.hip).
#pragma once
#include "dl_common.h"

struct DwnRows {
    const float *x, *thr;        // the layer's input: x [B][I], the features [B][I / nbits] whose code it is (thr),
    const uint8_t *planes;       // or bit-planes
    const int *idx32;
    const float *luts;
    float *y;                    // [B][NO], or null
    uint8_t *planes_out;         // the output as bit-planes, or null
    float *logits;               // [B][groups] sums, or null (then alone)
    uint8_t *saved;              // the addresses for a backward; null: inference, where the output is (table entry >= 0.5)
    int B, I, N, O, nbits, groups, gsize;
    float inv_tau;
};
// k <= DL_MAX_FAST_K
void dwn_launch_rows(int k, const DwnRows &a, hipStream_t s);
// us of that launch under a head, and whether it is the better one for a layer that writes planes: width features or values of x with
// nbits columns each, 0 planes in; up to DL_DWN_ROWS_INPUTS inputs
double dwn_rows_us(int B, int width, int nbits, int NO, int k, int groups, bool training);
bool dwn_rows_planes_pay(int B, int width, int nbits, int NO, bool training);
