// Rect tiles of a wave's 64 primitives as one task list spread over the
// wave's lanes (the preprocess's exact tile count and the instance emission).
//
// Task t < sum of the rect sizes is rect tile t - ex[j] (row major in the
// rect) of lane j's primitive, ex the exclusive prefix of the rect sizes.
// Each window of 64 consecutive tasks runs one per lane, whatever the sizes,
// so neither large nor uneven small rects leave lanes idle. The owner j of a
// task is the last lane whose rect starts at or before it: every rect that
// starts inside the window marks its start position in LDS, and a prefix
// maximum over the window, carrying the previous window's last owner, spreads
// the marks. The owner's values then come over ds_bpermute.
//
// A rect of more than kBigRect tiles is walked by the whole wave instead, 64
// tiles per step: its values are wave-uniform (scalar registers), so nothing
// is gathered or marked, and its hits are counted by ballot.
#pragma once
#include "common.h"

namespace tgs {

__device__ __forceinline__ uint32_t wave_inclusive_max_u32(uint32_t v) {
    v = max(v, dpp_u32<0x111>(v));          // row_shr:1
    v = max(v, dpp_u32<0x112>(v));          // row_shr:2
    v = max(v, dpp_u32<0x114>(v));          // row_shr:4
    v = max(v, dpp_u32<0x118>(v));          // row_shr:8
    v = max(v, dpp_u32<0x142, 0xA>(v));     // row_bcast:15
    v = max(v, dpp_u32<0x143, 0xC>(v));     // row_bcast:31
    return v;
}

// lane j's value of v (every lane of the wave must execute the call)
__device__ __forceinline__ uint32_t lane_gather(uint32_t j, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(j << 2), (int)v);
}

// Owner lane of task base + lane. nrect, ex: this lane's rect size and
// exclusive prefix; s_mark: 64 words of this wave's LDS; carry: 1 + the
// owner of the previous window's last task (0 before the first window),
// updated for the next window. Called by the whole wave.
__device__ __forceinline__ uint32_t wave_task_owner(uint32_t* s_mark, uint32_t nrect, uint32_t ex, uint32_t base,
                                                    uint32_t& carry) {
    const uint32_t lane = lane_id();
    s_mark[lane] = 0u;
    wave_lds_sync();
    if (nrect > 0u && ex >= base && ex - base < (uint32_t)kWave) s_mark[ex - base] = lane + 1u;
    wave_lds_sync();
    const uint32_t j = max(wave_inclusive_max_u32(s_mark[lane]), carry) - 1u;
    carry = readlane_u32(j, 63) + 1u;
    return j;
}

// (column, row) of rect tile k in a rect of width w: k / w through a float
// reciprocal. k < 2^16 and w <= 2^16 (grids are at most 2^16 tiles) are exact
// floats, and the estimate is off by at most one, corrected once.
__device__ __forceinline__ void rect_tile_of(uint32_t k, uint32_t w, uint32_t& col, uint32_t& row) {
    uint32_t q = (uint32_t)((float)k * __builtin_amdgcn_rcpf((float)w));
    int32_t r = (int32_t)k - (int32_t)(q * w);
    if (r < 0) {
        --q;
        r += (int32_t)w;
    } else if (r >= (int32_t)w) {
        ++q;
        r -= (int32_t)w;
    }
    col = (uint32_t)r;
    row = q;
}

// Rects of more tiles than this are walked one by one. The emission record holds
// the preprocess's outcomes of up to 32 tiles, so the emission's task list then
// needs no tile test; a walk of one step costs less than half a window of tasks,
// which puts the break-even at about half a step, 32 tiles, as well.
constexpr uint32_t kBigRect = 32u;

// Calls step(valid, tile x, tile y) for the tiles of one big rect, 64 per step in
// lane order; the arguments are wave-uniform, n > 0 (tested at the bottom of the
// loop: 345 -> 334 us in the preprocess of 375k primitives of about 200 tiles).
// Columns and rows advance by 64 / w and 64 % w, exact for any rect.
template <class Step>
__device__ __forceinline__ void walk_big_rect(uint32_t n, uint32_t org, uint32_t w, Step step) {
    uint32_t col, row, dcol, drow;
    rect_tile_of(lane_id(), w, col, row);
    rect_tile_of((uint32_t)kWave, w, dcol, drow);
    uint32_t first = 0;
    do {
        step(first + lane_id() < n, (org & 0xffffu) + col, (org >> 16) + row);
        first += (uint32_t)kWave;
        col += dcol;
        row += drow;
        if (col >= w) {
            col -= w;
            ++row;
        }
    } while (first < n);
}

// RN(a / b) for y = RN(1 / b), or by division where y is 0: two residual
// corrections of a y (P. Markstein, "Computation of elementary functions on
// the IBM RISC System/6000 processor", 1990: the second starts within one unit
// in the last place of the quotient, so it rounds correctly). y is 0 unless
// 2^-40 <= |b| <= 2^40 (tile_test_inverse) and |a| is checked here, so no
// residual or quotient leaves the normal range. Five operations instead of the
// division's eleven.
TGS_HD float quotient_by(float a, float b, float y) {
    const float m = __builtin_fabsf(a);
    if (!(y != 0.0f && m >= 0x1p-60f && m <= 0x1p60f)) return a / b;
    float q = a * y;
    q = __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
    return __builtin_fmaf(__builtin_fmaf(-b, q, a), y, q);
}

// The divisor of the tile test along an axis with conic diagonal c: (dx c) dx
// for dx = +-15, the same value for both signs; and its reciprocal as
// quotient_by takes it.
TGS_HD float tile_test_divisor(float c) { return (15.0f * c) * 15.0f; }
TGS_HD float tile_test_inverse(float c) {
    const float b = tile_test_divisor(c), m = __builtin_fabsf(b);
    return m >= 0x1p-40f && m <= 0x1p40f ? 1.0f / b : 0.0f;
}

// kernels_forward.cuh:49-84, on the mean shifted by -0.5 (:94): whether the
// primitive may contribute to a tile. ia, ic: tile_test_inverse of ca and cc.
__device__ __forceinline__ bool will_contribute(float mx, float my, float ca, float cb, float cc, float ia, float ic,
                                                uint32_t tile_x, uint32_t tile_y, float power_threshold) {
    const float rminx = (float)(tile_x * 16u), rminy = (float)(tile_y * 16u);
    const float rmaxx = rminx + 15.0f, rmaxy = rminy + 15.0f;
    const float x_min_diff = rminx - mx, y_min_diff = rminy - my;
    const bool left = x_min_diff > 0.0f, above = y_min_diff > 0.0f;
    const bool out_x = left || mx > rmaxx, out_y = above || my > rmaxy;
    // the tile corner nearest the mean
    const float ccx = left ? rminx : rmaxx, ccy = above ? rminy : rmaxy;
    const float diffx = mx - ccx, diffy = my - ccy;
    const float dx = __builtin_copysignf(15.0f, x_min_diff);
    const float dy = __builtin_copysignf(15.0f, y_min_diff);
    const float qx = quotient_by(dx * ca * diffx + dx * cb * diffy, tile_test_divisor(ca), ia);
    const float qy = quotient_by(dy * cb * diffx + dy * cc * diffy, tile_test_divisor(cc), ic);
    const float tx = out_y ? saturate(qx) : 0.0f, ty = out_x ? saturate(qy) : 0.0f;
    const float px = ccx + tx * dx, py = ccy + ty * dy;
    const float ddx = mx - px, ddy = my - py;
    const float max_power = 0.5f * (ca * ddx * ddx + cc * ddy * ddy) + cb * ddx * ddy;
    return !(out_x || out_y) || max_power <= power_threshold;
}

}  // namespace tgs
