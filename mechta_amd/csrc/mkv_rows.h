// mkv_rows.h -- conversion between the reference's position-major rows ([pos][kv head][dim], 512 elements a position) and
// the store's planes, 16 positions per work-group, for both models (2 heads of 256 dims, 4 heads of 128).
//
// The conversion moves each byte once, so HBM (and below a few thousand positions the launch) bounds it; what kept the
// one-element-per-thread kernel from that were 2-byte accesses 16 bytes apart. 8,192 positions of f16 K and V read out,
// written into another store and read again (six conversions of 16.8 MB): 56.4 us with it, 24.8 us here (4.1 TB/s).
// Every global access is 16 bytes per lane, in runs of 64 bytes or more on both sides:
//   K: a 16-byte chunk is consecutive dims of one position on both sides, so it only moves; a wave takes 16 positions x
//      4 chunks (256-byte runs in the plane, 64-byte runs in the rows);
//   V: a chunk holds 8 (f16) or 4 (f32) positions of one dim, so the 16 positions pass through LDS.
// Rows that are not 16-byte aligned keep the element kernel.
#pragma once
#include "mkv_internal.h"

namespace mkv {
namespace rows {

constexpr int PB = 16;    // positions per work-group
constexpr int ROWE = 512; // elements of a position
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// E: unsigned short or float; DIR 0: planes -> rows, 1: rows -> planes. plane: kv head 0's plane, the heads plane_elems
// apart; rows: position p0 first; positions [p0, p1).
template <typename E, int HD, int DIR, int WHICH>
__global__ void __launch_bounds__(256) rows_tile(E* __restrict__ plane, size_t plane_elems, E* __restrict__ rows, int p0,
                                                 int p1) {
    constexpr int EPC = 16 / sizeof(E);          // elements of a chunk
    constexpr int CPR = ROWE / EPC;              // chunks of a row
    constexpr int IT = PB * CPR / 256;           // chunks per thread: 4 (f16) or 8 (f32)
    const int tid = threadIdx.x;
    const int q0 = (p0 / PB + blockIdx.x) * PB;  // the work-group's positions [q0, q0 + PB), cut to [p0, p1)
    if constexpr (WHICH == 0) {
        u32x4 x[IT];
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const int c = tid + 256 * k, p = q0 + (c & (PB - 1)), e = (((c >> 6) << 2) | ((c >> 4) & 3)) * EPC;
            const int kh = e / HD, d = e % HD;
            const size_t po = (size_t)kh * plane_elems + (size_t)(p / KBLK) * (KBLK * HD) + (size_t)(d / EPC) * (KBLK * EPC) +
                              (size_t)(p % KBLK) * EPC;
            if (p >= p0 && p < p1)
                x[k] = DIR == 0 ? *(const u32x4*)(plane + po) : *(const u32x4*)(rows + (size_t)(p - p0) * ROWE + e);
        }
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const int c = tid + 256 * k, p = q0 + (c & (PB - 1)), e = (((c >> 6) << 2) | ((c >> 4) & 3)) * EPC;
            const int kh = e / HD, d = e % HD;
            const size_t po = (size_t)kh * plane_elems + (size_t)(p / KBLK) * (KBLK * HD) + (size_t)(d / EPC) * (KBLK * EPC) +
                              (size_t)(p % KBLK) * EPC;
            if (p >= p0 && p < p1) {
                if (DIR == 0) *(u32x4*)(rows + (size_t)(p - p0) * ROWE + e) = x[k];
                else *(u32x4*)(plane + po) = x[k];
            }
        }
    } else {
        // V: group = EPC positions of every dim; the tile in LDS position-major
        __shared__ __attribute__((aligned(16))) E t[PB][ROWE];
        constexpr int NG = PB / EPC;
        auto group = [&](int g, int e) { return plane + (size_t)(e / HD) * plane_elems + (size_t)(q0 / EPC + g) * (EPC * HD) + (size_t)(e % HD) * EPC; };
        if constexpr (DIR == 1) {
            // rows outside the range are loaded as its nearest one and not stored: a load behind a branch each took the f32
            // build to 230 registers and one load at a time (100 positions 4.5 us, 1,000 4.8; now 2.3 and 2.6)
            u32x4 x[IT];
#pragma unroll
            for (int k = 0; k < IT; k++) {
                const int c = tid + 256 * k, p = min(max(q0 + c / CPR, p0), p1 - 1), e = (c % CPR) * EPC;
                x[k] = *(const u32x4*)(rows + (size_t)(p - p0) * ROWE + e);
            }
#pragma unroll
            for (int k = 0; k < IT; k++) {
                const int c = tid + 256 * k;
                *(u32x4*)&t[c / CPR][(c % CPR) * EPC] = x[k];
            }
            __syncthreads();
#pragma unroll
            for (int g = 0; g < NG; g++) {
                const int a = max(q0 + g * EPC, p0), b = min(q0 + (g + 1) * EPC, p1);
                if (a >= b) continue;
                if constexpr (sizeof(E) == 2) {  // two dims per thread: 8 LDS words, two chunks
                    unsigned w[8];
#pragma unroll
                    for (int i = 0; i < 8; i++) w[i] = *(const unsigned*)&t[g * EPC + i][2 * tid];
                    if (b - a == EPC) {
                        u32x4 lo, hi;
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            lo[i] = (w[2 * i] & 0xffffu) | w[2 * i + 1] << 16;
                            hi[i] = w[2 * i] >> 16 | (w[2 * i + 1] & 0xffff0000u);
                        }
                        u32x4* o = (u32x4*)group(g, 2 * tid);
                        o[0] = lo;
                        o[1] = hi;
                    } else {  // a group that [p0, p1) covers in part: its other positions stay
                        E* o = group(g, 2 * tid);
#pragma unroll
                        for (int i = 0; i < 8; i++) {
                            const int p = q0 + g * EPC + i;
                            if (p >= a && p < b) {
                                o[i] = (E)(w[i] & 0xffffu);
                                o[EPC + i] = (E)(w[i] >> 16);
                            }
                        }
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        const int e = tid + 256 * k;
                        E* o = group(g, e);
                        if (b - a == EPC) {
                            *(float4*)o = make_float4(t[g * EPC][e], t[g * EPC + 1][e], t[g * EPC + 2][e], t[g * EPC + 3][e]);
                        } else {
                            for (int p = a; p < b; p++) o[p - q0 - g * EPC] = t[p - q0][e];
                        }
                    }
                }
            }
        } else {
            // the plane's chunks (whole groups: the plane holds every position of a group), then the rows
#pragma unroll
            for (int g = 0; g < NG; g++) {
                if constexpr (sizeof(E) == 2) {
                    const u32x4* o = (const u32x4*)group(g, 2 * tid);
                    const u32x4 lo = o[0], hi = o[1];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        *(unsigned*)&t[g * EPC + 2 * i][2 * tid] = (lo[i] & 0xffffu) | hi[i] << 16;
                        *(unsigned*)&t[g * EPC + 2 * i + 1][2 * tid] = lo[i] >> 16 | (hi[i] & 0xffff0000u);
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        const int e = tid + 256 * k;
                        const float4 x = *(const float4*)group(g, e);
                        t[g * EPC][e] = x.x;
                        t[g * EPC + 1][e] = x.y;
                        t[g * EPC + 2][e] = x.z;
                        t[g * EPC + 3][e] = x.w;
                    }
                }
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < IT; k++) {
                const int c = tid + 256 * k, p = q0 + c / CPR, e = (c % CPR) * EPC;
                if (p >= p0 && p < p1) *(u32x4*)(rows + (size_t)(p - p0) * ROWE + e) = *(const u32x4*)&t[c / CPR][e];
            }
        }
    }
}

template <typename E, int HD>
hipError_t launch_tile(E* plane, size_t plane_elems, E* rows, int which, int p0, int p1, int dir, const Launch& L) {
    const dim3 grid((p1 - 1) / PB - p0 / PB + 1);
    auto k = which == 0 ? (dir == 0 ? rows_tile<E, HD, 0, 0> : rows_tile<E, HD, 1, 0>)
                        : (dir == 0 ? rows_tile<E, HD, 0, 1> : rows_tile<E, HD, 1, 1>);
    return launch(k, grid, dim3(256), L, plane, plane_elems, rows, p0, p1);
}

}  // namespace rows
}  // namespace mkv
