// Channels of particle state between particle order and an engine's slot order: dst[c][to(i)] = src[c][from(i)].
//
// One thread per particle moves a particle's channels one by one.  While neighbouring slots hold
// neighbouring particles (a lattice scene, also when it has moved for some time) its scattered 4-byte
// accesses share cache lines and it runs at the copy rate.  Once particles have mixed, or an image's
// particles come in no order, every access takes a line of its own: 25 channels of 1,048,576 particles
// in 496 us.  Large sets then go through rows instead: the channels are transposed through LDS into one
// row per particle, the rows are moved as a whole (a line or two each) and transposed back: 83 + 70 us,
// whatever the order (in order the direct form takes 47).  Which of the two runs is decided on the device,
// from how many neighbouring entries of the order fall into other cache lines, since the host does
// not know the order; the other's workgroups end at once.
//
// A large state image is also stored in tile order when it is set (its copy has to be written anyway)
// by a caller that leaves the slot order to the engine, so that the first step reads it in order: P2G and G2P of 1,048,576 particles in random order took
// 506 and 296 us there instead of 139 and 99.  Six steps from such an image, the image in and out:
// 3.13 -> 2.37 ms.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mpm_device.hpp"

namespace nclr_dev {

// One workgroup looks at kSamples runs of 64 entries, evenly spread over an order; an entry changes line
// where its 32-entry line is not its predecessor's.  Rows are faster beyond a quarter (in order: one
// in 32 to one in 8; at random: all).
constexpr int kSamples = 256;
NCLR_DI bool by_rows(const uint32_t* __restrict__ changes) { return *changes > kSamples * 64 / 4; }

__global__ __launch_bounds__(1024) void k_line_changes(const uint32_t* __restrict__ order, int64_t n,
                                                       uint32_t* __restrict__ changes) {
    __shared__ uint32_t s_count[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t line[kSamples / 16], mine = 0;
#pragma unroll
    for (int r = 0; r < kSamples / 16; ++r) {
        const int64_t i = (n - 64) * (r * 16 + wave) / (kSamples - 1) + lane;  // n >= 64
        line[r] = order[i] >> 5;
    }
#pragma unroll
    for (int r = 0; r < kSamples / 16; ++r) {
        const uint32_t before = __shfl_up(line[r], 1);
        mine += uint32_t(__popcll(__ballot(lane > 0 && line[r] != before)));
    }
    if (lane == 0) s_count[wave] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t sum = 0;
        for (int w = 0; w < 16; ++w) sum += s_count[w];
        *changes = sum;
    }
}

// dst[c][to(i)] = src[c][from(i)]: with to_particle_order, slot i goes to particle pid[i];
// otherwise slot i takes particle pid[i].  changes (or nullptr): only if the order is not to go by rows.
__global__ __launch_bounds__(256) void k_permute_channels(const uint32_t* __restrict__ pid, const float* __restrict__ src,
                                                          int64_t src_stride, float* __restrict__ dst,
                                                          int64_t dst_stride, int channels, int64_t n,
                                                          int to_particle_order, const uint32_t* __restrict__ changes) {
    if (changes && by_rows(changes)) return;
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t u = pid[i];
    const int64_t si = to_particle_order ? i : u;
    const int64_t di = to_particle_order ? u : i;
    for (int c = 0; c < channels; ++c) dst[int64_t(c) * dst_stride + di] = src[int64_t(c) * src_stride + si];
}

// 64 particles at a time per workgroup (at most 4,096 workgroups, which end
// within 3 us when the rows are not taken; 1,024 cannot keep the loads in flight: 117 us against 77):
// channel c of particle i at src[c * src_stride + i] -> row at(i) = order[i] (or i) of
// `channels` floats.
constexpr int kRowParticles = 64;
constexpr int kMaxRow = 27;
__global__ __launch_bounds__(256) void k_channels_to_rows(const uint32_t* __restrict__ order, const float* __restrict__ src,
                                                          int64_t src_stride, float* __restrict__ rows, int channels,
                                                          int64_t n, const uint32_t* __restrict__ changes) {
    __shared__ float t[kRowParticles][kMaxRow + 2];
    if (!by_rows(changes)) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int64_t i0 = int64_t(blockIdx.x) * kRowParticles; i0 < n; i0 += int64_t(gridDim.x) * kRowParticles) {
        for (int c = wave; c < channels; c += 4)
            if (i0 + lane < n) t[lane][c] = src[int64_t(c) * src_stride + i0 + lane];
        __syncthreads();
        for (int e = threadIdx.x; e < kRowParticles * channels; e += 256) {
            const int q = e / channels, c = e - q * channels;
            if (i0 + q < n) rows[int64_t(order ? order[i0 + q] : uint32_t(i0 + q)) * channels + c] = t[q][c];
        }
        __syncthreads();
    }
}

// The way back: row order[j] (or j) -> channels at j.
__global__ __launch_bounds__(256) void k_rows_to_channels(const uint32_t* __restrict__ order, const float* __restrict__ rows,
                                                          float* __restrict__ dst, int64_t dst_stride, int channels,
                                                          int64_t n, const uint32_t* __restrict__ changes) {
    __shared__ float t[kRowParticles][kMaxRow + 2];
    if (!by_rows(changes)) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int64_t j0 = int64_t(blockIdx.x) * kRowParticles; j0 < n; j0 += int64_t(gridDim.x) * kRowParticles) {
        for (int e = threadIdx.x; e < kRowParticles * channels; e += 256) {
            const int q = e / channels, c = e - q * channels;
            if (j0 + q < n) t[q][c] = rows[int64_t(order ? order[j0 + q] : uint32_t(j0 + q)) * channels + c];
        }
        __syncthreads();
        for (int c = wave; c < channels; c += 4)
            if (j0 + lane < n) dst[int64_t(c) * dst_stride + j0 + lane] = t[lane][c];
        __syncthreads();
    }
}

// The tile keys of a state image (particle order, n floats per row): k_keys without the step's stamp, and a
// scene with a particle off its grid only noted (the step that follows reports and stops it).
template <int D>
__global__ __launch_bounds__(256) void k_image_keys(const float* __restrict__ image, StepParams p,
                                                    uint32_t* __restrict__ keys, uint32_t* __restrict__ tile_start,
                                                    uint32_t* __restrict__ tile_end, uint32_t* __restrict__ off_grid) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i <= int64_t(p.ntiles)) {
        tile_start[i] = 0;
        tile_end[i] = 0;
    }
    if (i >= p.n) return;
    const int s = p.nscenes == 1 ? 0 : scene_of_particle(p, uint32_t(i));
    const SceneParams sp = p.scenes[s];
    float x[D];
#pragma unroll
    for (int a = 0; a < D; ++a) x[a] = image[int64_t(Layout<D>::X + a) * p.n + i];
    int base[D];
    float fx[D], w[D][3];
    if (stencil<D>(x, sp, base, fx, w)) {
        keys[i] = sp.tile_base + tile_key<D>(base, sp.nt);
    } else {
        keys[i] = p.ntiles;
        off_grid[s] = 1u;
    }
}

// mass and volume of slot i to particle pid[i]
__global__ __launch_bounds__(256) void k_constants_to_particles(const uint32_t* __restrict__ pid,
                                                                const float* __restrict__ mass,
                                                                const float* __restrict__ vol, float* __restrict__ mass_p,
                                                                float* __restrict__ vol_p, int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    mass_p[pid[i]] = mass[i];
    vol_p[pid[i]] = vol[i];
}

// Slot j of the state takes particle perm[j] of the image; the constants and the slot -> particle map
// always here (the rows are moved by that map), the channels unless they go by rows.  The slots
// are then in sorted order: perm becomes the identity.
__global__ __launch_bounds__(256) void k_image_to_slots(uint32_t* __restrict__ perm, const float* __restrict__ image,
                                                        const float* __restrict__ mass_p, const float* __restrict__ vol_p,
                                                        float* __restrict__ st, uint32_t* __restrict__ pid,
                                                        int64_t stride, int channels, int64_t n,
                                                        const uint32_t* __restrict__ changes) {
    const int64_t j = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const uint32_t i = perm[j];
    perm[j] = uint32_t(j);
    pid[j] = i;
    st[int64_t(channels) * stride + j] = mass_p[i];
    st[int64_t(channels + 1) * stride + j] = vol_p[i];
    if (by_rows(changes)) return;
    for (int c = 0; c < channels; ++c) st[int64_t(c) * stride + j] = image[int64_t(c) * n + i];
}

// Stops the scenes with a particle off their grid, ahead of an incremental sort from a sorted image: the sort
// finds such particles itself, but in the launch that lists the node tiles, which leaves a stopped
// scene's counts as they are.
__global__ __launch_bounds__(256) void k_stop_off_grid(StepParams p, const uint32_t* __restrict__ off_grid) {
    const int64_t s = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (s < p.nscenes && off_grid[s]) stop_scene(p, int(s), kStatusOutOfRange);
}

// The sort of the step after a sorted image: the slots are in order and the tables stand; the step's stamp,
// the scenes with a particle off their grid and the node tiles are left to do.
template <int D>
__global__ __launch_bounds__(256) void k_sorted_step(StepParams p, uint32_t* __restrict__ stamp,
                                                     const uint32_t* __restrict__ off_grid,
                                                     const uint32_t* __restrict__ item_offset,
                                                     GridTile<D>* __restrict__ tiles, uint32_t* meta,
                                                     uint32_t* __restrict__ active) {
    const int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (t == 0) *stamp = *stamp + 1u;
    if (t < p.nscenes && off_grid[t]) stop_scene(p, int(t), kStatusOutOfRange);
    const bool stops = t < p.node_tiles && off_grid[p.nscenes == 1 ? 0 : scene_of_node_tile(p, uint32_t(t))] != 0u;
    list_grid_tile<D>(p, stops ? p.node_tiles : uint32_t(t), item_offset, tiles, &meta[kMetaGridTiles], active);
}

// order[j] = the particle of sorted position j.
__global__ __launch_bounds__(256) void k_sorted_order(const uint32_t* __restrict__ pid, const uint32_t* __restrict__ perm,
                                                      uint32_t* __restrict__ order, int64_t n) {
    const int64_t j = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (j < n) order[j] = pid[perm[j]];
}

// Slots -> particle-major arrays in particle order, for the host: the device does the reordering and the
// transposition, so that the host only copies.
template <int D>
__global__ __launch_bounds__(256) void k_particles_out(const float* __restrict__ st, const uint32_t* __restrict__ pid,
                                                       int64_t n, int64_t stride, float* __restrict__ out) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t to = pid[i];
    if (to >= n) return;
    int row = 0;
    auto put = [&](auto width) {
        constexpr int K = decltype(width)::value;
#pragma unroll
        for (int k = 0; k < K; ++k) out[row * n + to * K + k] = st[(row + k) * stride + i];
        row += K;
    };
    using std::integral_constant;
    put(integral_constant<int, D>{});      // x
    put(integral_constant<int, D>{});      // v
    put(integral_constant<int, D * D>{});  // F
    put(integral_constant<int, D * D>{});  // C
    put(integral_constant<int, 1>{});      // Jp
    put(integral_constant<int, 1>{});      // mass
    put(integral_constant<int, 1>{});      // volume
}

}  // namespace nclr_dev

namespace nclr_host {

using namespace nclr_dev;

static inline unsigned blocks_of(int64_t n, int threads) { return unsigned((n + threads - 1) / threads); }
static unsigned row_blocks(int64_t n) { return unsigned(std::min<int64_t>((n + kRowParticles - 1) / kRowParticles, 4096)); }

// Below this count the set fits the L2 caches and the direct form is as fast in any order (150,003
// particles at random: 36 us, by rows 23 and the two launches that decide).
constexpr int64_t kMinByRows = int64_t(1) << 18;
// A sorted image's first step lists the node tiles: launches of that size do (grid_tiles_listed).
static_assert(kMinByRows >= int64_t(kFewItems) * kMaxChunk, "sorted images have listed node tiles");

hipError_t launch_permute_channels(const uint32_t* pid, const float* src, int64_t src_stride, float* dst,
                                   int64_t dst_stride, int channels, int64_t n, bool to_particle_order, float* rows,
                                   uint32_t* changes, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    const bool choose = rows && n >= kMinByRows && channels <= kMaxRow;
    if (choose) {
        k_line_changes<<<1, 1024, 0, s>>>(pid, n, changes);
    }
    k_permute_channels<<<blocks_of(n, 256), 256, 0, s>>>(pid, src, src_stride, dst, dst_stride, channels, n,
                                                         to_particle_order ? 1 : 0, choose ? changes : nullptr);
    if (choose) {
        const unsigned b = row_blocks(n);
        k_channels_to_rows<<<b, 256, 0, s>>>(to_particle_order ? pid : nullptr, src, src_stride, rows, channels, n,
                                             changes);
        k_rows_to_channels<<<b, 256, 0, s>>>(to_particle_order ? nullptr : pid, rows, dst, dst_stride, channels, n,
                                             changes);
    }
    return hipGetLastError();
}

hipError_t launch_stop_off_grid(const LaunchArgs& a) {
    k_stop_off_grid<<<blocks_of(a.p.nscenes, 256), 256, 0, a.stream>>>(a.p, a.off_grid);
    return hipGetLastError();
}

hipError_t launch_sorted_step(const LaunchArgs& a) {
    const unsigned b = std::max(1u, blocks_of(std::max<int64_t>(a.p.node_tiles, a.p.nscenes), 256));
    if (a.dim == 2)
        k_sorted_step<2><<<b, 256, 0, a.stream>>>(a.p, a.stamp, a.off_grid, a.item_offset,
                                                  static_cast<GridTile<2>*>(a.grid_tiles), a.meta, a.active);
    else
        k_sorted_step<3><<<b, 256, 0, a.stream>>>(a.p, a.stamp, a.off_grid, a.item_offset,
                                                  static_cast<GridTile<3>*>(a.grid_tiles), a.meta, a.active);
    return hipGetLastError();
}

hipError_t launch_particles_out(int dim, const float* st, const uint32_t* pid, int64_t n, int64_t stride, float* out,
                                hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (dim == 2) k_particles_out<2><<<blocks_of(n, 256), 256, 0, s>>>(st, pid, n, stride, out);
    else k_particles_out<3><<<blocks_of(n, 256), 256, 0, s>>>(st, pid, n, stride, out);
    return hipGetLastError();
}

hipError_t launch_sorted_order(const LaunchArgs& a, uint32_t* order) {
    if (a.p.n <= 0) return hipSuccess;
    k_sorted_order<<<blocks_of(a.p.n, 256), 256, 0, a.stream>>>(a.pid_in, a.perm, order, a.p.n);
    return hipGetLastError();
}

bool image_goes_sorted(int64_t n) { return n >= kMinByRows; }

hipError_t launch_image_keys(const LaunchArgs& a, const float* image, uint32_t* keys) {
    const unsigned b = blocks_of(std::max<int64_t>(a.p.n, int64_t(a.p.ntiles) + 1), 256);
    const hipError_t e = launch_fill_u32(a.off_grid, a.p.nscenes, 0u, a.stream);
    if (e != hipSuccess) return e;
    if (a.dim == 2) k_image_keys<2><<<b, 256, 0, a.stream>>>(image, a.p, keys, a.tile_start, a.tile_end,
                                                                a.off_grid);
    else k_image_keys<3><<<b, 256, 0, a.stream>>>(image, a.p, keys, a.tile_start, a.tile_end,
                                                                a.off_grid);
    return hipGetLastError();
}

hipError_t launch_image_to_slots(const LaunchArgs& a, const float* image, int channels, float* st, uint32_t* pid,
                                 uint32_t* changes) {
    const int64_t n = a.p.n, stride = a.p.stride;
    const unsigned b = blocks_of(n, 256);
    hipStream_t s = a.stream;
    // the sort's temporaries hold the particles' constants, the old state (its constants read) the rows
    float *mass_p = reinterpret_cast<float*>(a.keys_tmp), *vol_p = reinterpret_cast<float*>(a.perm_tmp);
    float* rows = const_cast<float*>(a.state_in);
    k_line_changes<<<1, 1024, 0, s>>>(a.perm, n, changes);
    k_constants_to_particles<<<b, 256, 0, s>>>(a.pid_in, a.state_in + int64_t(channels) * stride,
                                               a.state_in + int64_t(channels + 1) * stride, mass_p, vol_p, n);
    k_image_to_slots<<<b, 256, 0, s>>>(a.perm, image, mass_p, vol_p, st, pid, stride, channels, n, changes);
    const unsigned rb = row_blocks(n);
    k_channels_to_rows<<<rb, 256, 0, s>>>(nullptr, image, n, rows, channels, n, changes);
    k_rows_to_channels<<<rb, 256, 0, s>>>(pid, rows, st, stride, channels, n, changes);
    return hipGetLastError();
}

}  // namespace nclr_host
