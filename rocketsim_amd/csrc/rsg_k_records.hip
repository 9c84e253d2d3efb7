// rsg_k_records.hip -- the public records (include/rsg_state.h) of a batch's
// cars, balls and pads, read from the word planes on the device, and the
// controls scattered into them.
//
// What bounds them: the trip over PCIe; the planes' words and the conversion
// are a small part.  Records are made in LDS, one car or ball (or one arena's
// pads) a lane, so that plane reads run along the arenas, and leave as whole
// lines of 16 bytes a lane straight into pinned host memory (2v2 x 16384
// arenas, 29 MB: 1.1 ms with the copies out of it).
#include <hip/hip_runtime.h>

#include "rsg_api_convert.h"
#include "rsg_kernels.h"

using namespace rsg;

namespace {

constexpr int LANES = 64;
constexpr int LOCAL_WORDS = LANES * PAD_NUM * (int)sizeof(rsg_pad_state) / 4;
static_assert(LOCAL_WORDS * 4 >= LANES * (int)sizeof(rsg_car_state) && LOCAL_WORDS * 4 >= LANES * (int)sizeof(rsg_ball_state),
              "the pads are the largest of the three");
static_assert(sizeof(rsg_pad_state) == 12 && sizeof(rsg_car_state) % 4 == 0 && sizeof(rsg_ball_state) % 4 == 0,
              "records are whole words");

// `bytes` of the local block to `out` (16-byte aligned: each block's share of
// a 16-byte aligned array is a multiple of 64 records).
__device__ void write_out(const uint32_t* local, void* out, int bytes) {
    const int quads = bytes / 16, words = bytes / 4;
    for (int i = threadIdx.x; i < quads; i += LANES)
        static_cast<uint4*>(out)[i] = reinterpret_cast<const uint4*>(local)[i];
    for (int i = quads * 4 + threadIdx.x; i < words; i += LANES) static_cast<uint32_t*>(out)[i] = local[i];
}

}  // namespace

__global__ void __launch_bounds__(LANES) rsg_records_read_kernel(BatchDev d, const int32_t* car_at, RecordsOut o) {
    __shared__ __align__(16) uint32_t local[LOCAL_WORDS];
    const int lane = threadIdx.x;
    int block = blockIdx.x;
    const int car_blocks = (o.n_cars + LANES - 1) / LANES, ball_blocks = (o.n_balls + LANES - 1) / LANES;
    if (block < car_blocks) {
        const int k = block * LANES + lane;
        if (k < o.n_cars) {
            const int at = car_at[o.first_car + k];
            car_to_api(car_ref(d, at >> 4, at & 15), reinterpret_cast<rsg_car_state*>(local)[lane]);
        }
        __syncthreads();
        write_out(local, o.cars + block * LANES, min(LANES, o.n_cars - block * LANES) * (int)sizeof(rsg_car_state));
        return;
    }
    block -= car_blocks;
    if (block < ball_blocks) {
        const int k = block * LANES + lane;
        if (k < o.n_balls)
            ball_to_api(ball_ref(d, o.first_ball + k), reinterpret_cast<rsg_ball_state*>(local)[lane]);
        __syncthreads();
        write_out(local, o.balls + block * LANES, min(LANES, o.n_balls - block * LANES) * (int)sizeof(rsg_ball_state));
        return;
    }
    block -= ball_blocks;
    const int k = block * LANES + lane;
    if (k < o.n_pad_arenas)
        for (int p = 0; p < PAD_NUM; p++)
            pad_to_api(pad_ref(d, o.first_pad_arena + k, p), reinterpret_cast<rsg_pad_state*>(local)[lane * PAD_NUM + p]);
    __syncthreads();
    write_out(local, o.pads + (size_t)block * LANES * PAD_NUM,
              min(LANES, o.n_pad_arenas - block * LANES) * PAD_NUM * (int)sizeof(rsg_pad_state));
}

// Controls from pinned host memory (16-byte aligned) into their words.
__global__ void __launch_bounds__(LANES) rsg_controls_write_kernel(BatchDev d, const int32_t* car_at,
                                                                   const rsg_controls* in, int n) {
    __shared__ __align__(16) uint32_t local[LANES * sizeof(rsg_controls) / 4];
    const int first = blockIdx.x * LANES, lane = threadIdx.x;
    const int words = min(LANES, n - first) * (int)sizeof(rsg_controls) / 4;
    const uint32_t* src = reinterpret_cast<const uint32_t*>(in + first);
    for (int i = lane; i < words; i += LANES) local[i] = src[i];
    __syncthreads();
    if (first + lane >= n) return;
    const int at = car_at[first + lane];
    store_ctrl(car_ref(d, at >> 4, at & 15), CW_CTRL, ctrl_from_api(reinterpret_cast<const rsg_controls*>(local)[lane]));
}

namespace rsg {

hipError_t launch_records_read(const BatchDev& d, const int32_t* car_at, const RecordsOut& o, hipStream_t s) {
    auto blocks = [](int n) { return (n + LANES - 1) / LANES; };
    const int grid = blocks(o.n_cars) + blocks(o.n_balls) + blocks(o.n_pad_arenas);
    if (grid == 0) return hipSuccess;
    rsg_records_read_kernel<<<grid, LANES, 0, s>>>(d, car_at, o);
    return hipGetLastError();
}

hipError_t launch_controls_write(const BatchDev& d, const int32_t* car_at, const rsg_controls* in, int n,
                                 hipStream_t s) {
    rsg_controls_write_kernel<<<(n + LANES - 1) / LANES, LANES, 0, s>>>(d, car_at, in, n);
    return hipGetLastError();
}

}  // namespace rsg
