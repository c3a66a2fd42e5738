// MHD constrained-transport stage passes (both precisions).
#include <algorithm>
#include "launch.hpp"

namespace m3p {

long mhd_workspace_bytes(int N, int precision)
{
    const long N3 = (long)N * N * N, nf = (long)(N + 1) * N * N;
    const long rs = precision == M3P_FP64 ? 8 : 4;
    // primitives [8 N^3] and face fields [2][nf] per family, the primitive
    // pass's speeds, dt, and the alignment of the first and the third
    return (8 * N3 + 3 * 2 * nf) * rs + 8 * kMhdPrimGroups + 8 + 2 * 256;
}

// The three states of an RK2 step (64 B a cell each) are larger than the
// 256 MB memory-side cache.  Non-temporal accesses then, for what a pass
// touches once: a step of 256^3 mixed 2625 us to 2470 (FP64 3995 to 3930),
// 160^3 664 to 616, 128^3 343 to 301 (553 to 530), 112^3 245 to 242 (407 to
// 394); below the line the next pass would find them in cache, and 100^3 took
// 201 us instead of 191 (332 instead of 313), 96^3 160 instead of 154.
static bool mhd_streams(int N) { return 3 * 64 * (long)N * N * N > 256l << 20; }

template<typename R, bool NT>
static int mhd_advance_as(MhdArgs a, char* work, hipStream_t s)
{
    const int N = a.N;
    const long N3 = (long)N * N * N, nf = (long)(N + 1) * N * N;
    auto align = [] (char* p) { return p + ((256 - (reinterpret_cast<uintptr_t>(p) & 255)) & 255); };
    auto P = reinterpret_cast<typename MhdPrim<R>::V*>(align(work));
    R* E1 = reinterpret_cast<R*>(P) + 8 * N3;
    R* E2 = E1 + 2 * nf;
    R* E3 = E2 + 2 * nf;
    a.vmax = reinterpret_cast<double*>(align(reinterpret_cast<char*>(E3 + 2 * nf)));
    if (!a.dt) a.dt = a.vmax + kMhdPrimGroups;
    const int gc = (int)((N3 + 255) / 256);
    a.nvmax = std::min(gc, kMhdPrimGroups);
    hipLaunchKernelGGL((mhd_prim_kernel<R, NT>), dim3(a.nvmax), dim3(256), 0, s, a, P);
    FaceE<R> fe{ E1, E2, E3, N, nf };
    // Column tiles of 8 x 32 columns: fluxes and the conserved update in one
    // pass (16 x 16 tiles 0 to 10 % slower at 64 to 256, 8 x 8 tiles 20 to
    // 40 %).  A workgroup marches TI planes after a warm-up of about one, so
    // a cube that fills the device takes long segments (FP64, 16 planes:
    // 4.36 ms a step at 256^3 against 4.45 with 8) and a small one as many
    // workgroups as it can give (FP64 64^3: 98 us a step with 2 planes, 236
    // with 16; mixed 100^3: 190 us with 8, 233 with 16).  Mixed keeps to 8
    // planes (1.37 ms at 200^3 against 1.42 with 16, equal at 256^3).
    const bool ragged = N % 32 != 0;
    const MhdTile tile = ragged && !NT ? mhd_ragged_tile(N) : kMhdWideTile;
    auto kern = ragged ? mhd_tile_kernel<R, true, false, NT> : mhd_tile_kernel<R, false, false, NT>;
    if constexpr (!NT) {
        if (tile.tj != kMhdWideTile.tj || tile.tk != kMhdWideTile.tk) kern = mhd_tile_kernel<R, true, true, NT>;
    }
    const int cols = ((N + tile.tj - 1) / tile.tj) * ((N + tile.tk - 1) / tile.tk);
    const int groups = is_fp64<R>::value ? 640 : 768, cap = is_fp64<R>::value ? 16 : 8;
    const int TI = (int)std::max(2l, std::min((long)cap, (long)N * cols / groups));
    hipLaunchKernelGGL(kern, dim3(cols * ((N + TI - 1) / TI)), dim3(kMhdTileLanes), 0, s, a,
                       (const typename MhdPrim<R>::V*)P, E1, E2, E3, TI, tile);
    if (int st = launch_status("mhd_tile_kernel")) return st;
    // The face fields: FP64 by bricks of 4 x 4 x 32 cells where they divide
    // the cube (the step 4.41 ms at 256^3 against 4.71 per cell, 626 us
    // against 672 at 128^3), else per cell (2.50 ms at 200^3 against 2.71 by
    // bricks of 2 x 4 x 8); mixed per cell, where the FP32 face fields that
    // the four faces of an edge re-read come from cache (bricks 0.5 % slower).
    if constexpr (is_fp64<R>::value) {
        if (N % 32 == 0) {
            hipLaunchKernelGGL((mhd_face_b_brick_kernel<R, 4, 4, 32, NT>), dim3((N / 4) * (N / 4) * (N / 32)), dim3(512),
                               0, s, a, fe);
            return launch_status("m3p_mhd_advance_ct");
        }
    }
    hipLaunchKernelGGL((mhd_face_b_kernel<R, NT>), dim3(gc), dim3(256), 0, s, a, fe);
    return launch_status("m3p_mhd_advance_ct");
}

template<typename R>
int mhd_advance(MhdArgs a, char* work, hipStream_t s)
{
    return mhd_streams(a.N) ? mhd_advance_as<R, true>(a, work, s) : mhd_advance_as<R, false>(a, work, s);
}

template int mhd_advance<double>(MhdArgs, char*, hipStream_t);
template int mhd_advance<float>(MhdArgs, char*, hipStream_t);

} // namespace m3p
