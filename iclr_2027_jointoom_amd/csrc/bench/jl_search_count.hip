// jl_search_count.hip - the row search's count of levels past a limit, with a
// limit of 40 cells instead of the frontier capacity.  A map that one
// wavefront searches has at most 16,384 cells, and no map of that size with
// a level of more than 4,096 of them is known, so the builder's own
// diagnostics cannot show this count at work on those layouts.  Built into
// libjl_bench.so; only its test loads it.
//
//   int jl_search_count(const uint32_t* map_bits, int32_t map_w, int32_t map_h,
//                       int32_t goal_x, int32_t goal_y, int32_t* count, jl_stream_t stream);
//
// count[0] = sum over the levels of the search from the goal (a free cell)
// of max(0, cells - 40).  Rows of 64, 96, 128 or 256 columns.
#include "../jl_bfs.h"

namespace jl {
namespace {

constexpr int kCountLimit = 40;

template <int H, int R, bool kSplit>
constexpr int count_waves() {
    return kSplit ? SearchShape<H, R>::kMaxWaves : 1;
}

template <int H, int R, bool kSplit>
__global__ __launch_bounds__((kWave * count_waves<H, R, kSplit>())) void search_count_kernel(
    const uint32_t* __restrict__ bits, int W, int gx, int gy, int32_t* __restrict__ count, int waves) {
    __shared__ SearchLds<H, R, kSplit, true, count_waves<H, R, kSplit>()> s;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int x0 = (kSplit ? wave * SearchShape<H, R>::kStep : 0) + lane * R;
    SearchPlanes<H, R, 1> P;
    load_search_rows<H, R>(bits, W, x0, P.avail);
    const int c = search_rows<H, R, kSplit, 1, 0, true, kCountLimit>(P, gx, gy, x0, lane, wave, waves, s, NoTallPlanes{});
    if (threadIdx.x == 0) count[0] = c;
}

template <int H>
int launch(const uint32_t* bits, int W, int gx, int gy, int32_t* count, hipStream_t stream) {
    const auto go = [&](auto kernel, int waves) {
        hipLaunchKernelGGL(kernel, dim3(1), dim3(kWave * waves), 0, stream, bits, W, gx, gy, count, waves);
        return launch_status();
    };
    // the layouts of the field searches: at most 8 words per lane, else split
    constexpr int kAlone = SearchShape<H, 4>::N <= 8 ? 4 : (SearchShape<H, 2>::N <= 8 ? 2 : 1);
    if (W <= kWave) return go(search_count_kernel<H, 1, false>, 1);
    if constexpr (kAlone >= 2)
        if (W <= 2 * kWave) return go(search_count_kernel<H, 2, false>, 1);
    if constexpr (kAlone == 4) return go(search_count_kernel<H, 4, false>, 1);
    else return go(search_count_kernel<H, kAlone, true>, split_waves<H, kAlone>(W));
}

}  // namespace
}  // namespace jl

using namespace jl;

extern "C" int jl_search_count(const uint32_t* map_bits, int32_t map_w, int32_t map_h, int32_t goal_x, int32_t goal_y,
                               int32_t* count, jl_stream_t stream) {
    if (!map_bits || !count || !profile_ok(map_w, map_h)) return JL_ERR_ARG;
    if (goal_x < 0 || goal_x >= map_w || goal_y < 0 || goal_y >= map_h) return JL_ERR_ARG;
    switch (map_h) {
        case 64: return launch<64>(map_bits, map_w, goal_x, goal_y, count, (hipStream_t)stream);
        case 96: return launch<96>(map_bits, map_w, goal_x, goal_y, count, (hipStream_t)stream);
        case 128: return launch<128>(map_bits, map_w, goal_x, goal_y, count, (hipStream_t)stream);
        case 256: return launch<256>(map_bits, map_w, goal_x, goal_y, count, (hipStream_t)stream);
        default: return JL_ERR_PROFILE;
    }
}
