// RnnKernel and RnnBackwardKernel (CX/kernels/rnn.h:34-66) for float32: every mode NStepRnnImpl hands to the kernel
// (CX/routines/n_step_rnn.cc:434-497) -- LSTM (mode 1), GRU (mode 0), plain RNN with tanh or relu (mode 2) -- in one or both
// directions, with the gradients of a forward pass that kept its reserve.
//
// The forward pass computes what the routine composition computes (GruImpl / LstmImpl / RnnImpl, n_step_rnn.cc:57-131; the layer
// and direction wiring of NStepRnnImpl, :362-426).  A time step of a layer-direction -- its products and its cells -- is one launch (RnnStepKernel), shared
// by all layer-directions that can advance at that point: both directions of a layer, or all layers of a one-directional network as a wavefront
// (layer l at step s - l).  Rows beyond a step's batch keep their state, as in OneDirectionalLoop (:133-175); the backward direction walks the
// steps from the last to the first on its own state.
//   * Small launches take the products with the layer's input along; else they are one product  XW = X_all [rows, in] . Wx^T  over the rows of
//     all steps of a layer (rows = sum of the steps' batch sizes).
//   * Large steps are a library product  h . Wh^T  and a launch of cells (Wide); so are their gradients.
//   * The state before a step is the output of the step before, where it lies; hy and cy are updated in place.
//   * The outputs go to columns [d*H, (d+1)*H) of the layer's output rows, which are the next layer's input (the Concatenate of
//     :398-404), or to the caller's ys[t] for the top layer.
// With a reserve (training) the steps also store what the gradient needs: the gate activations, the state rows before the
// step, and the outputs of the lower layers.  Large one-direction LSTMs without reserve are handed to hipcx_n_step_lstm (lstm.hip).
//
// The backward pass is backpropagation through time written out over the same buffers, the same layer-directions together: per step one
// cell-gradient kernel (gate pre-activation gradients from dh, dc, dy and the saved activations) and one launch of products (RnnBackKernel: with Wh for
// dh of the step before; in a wavefront with Wx too, for dy of the layer below); per layer
// and direction the weight gradients as products over all rows at once (dWx[g] = dG[:, g]^T . X_all, dWh[g] = dG[:, g]^T . Hprev_all),
// the bias gradients as column sums, and the input gradient dX_all = dG . Wx of the lowest layer (without a wavefront of every layer).
// The reference's cuda backend gets these numbers from cuDNN (CX/cuda/cuda_device/rnn.cu); every other backend from autograd over the
// composition.  Sums run in another order than either: equal to float32 tolerance.
#include <algorithm>
#include <utility>
#include <vector>

#include "common.h"
#include "dot_parts.h"
#include "small_dot.h"

extern "C" {
size_t hipcx_n_step_lstm_workspace_size(int n_layers, const hipcx_array* hx, const hipcx_array* const* xs, int n_steps);
int hipcx_n_step_lstm(int n_layers, const hipcx_array* hx, const hipcx_array* cx, const hipcx_array* const* ws, const hipcx_array* const* bs,
                      const hipcx_array* const* xs, int n_steps, const hipcx_array* hy, const hipcx_array* cy, const hipcx_array* const* ys,
                      void* workspace, size_t workspace_bytes, void* stream);
}

namespace hipcx {
namespace {

enum RnnMode { kGru = 0, kLstm = 1, kRnn = 2 };  // the `mode` argument of RnnKernel::Call as NStepRnnImpl's callers pass it

int NumGates(int mode) { return mode == kLstm ? 4 : (mode == kGru ? 3 : 1); }        // matrices per side; ws holds twice as many
int ReserveGates(int mode) { return mode == kRnn ? 1 : 4; }  // saved values per unit and row: LSTM i f g o; GRU r z n hh; RNN h

__device__ __forceinline__ float Sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }  // CX/routines/activation.cc:74-78

// Keeps a value that is the same for all lanes in scalar registers from here on.  Kernel arguments are otherwise fetched where they are first used, one
// dependent round trip to memory after the other; pinned together they come in one.
template <typename... T>
__device__ __forceinline__ void Pin(const T&... values) {
    (..., [](const auto& v) { asm volatile("" ::"s"(v)); }(values));
}

constexpr int kMaxJobs = 4;    // layer-directions that a launch advances by a step; their descriptors travel as kernel arguments
constexpr int kStepWaves = 8;  // per workgroup; they split the reduction
constexpr int kChunk = 32;     // terms of it that a wave takes at a time: a line of 128 bytes per row
constexpr int kPitch = 4 * kChunk + 16;  // bytes of a staged row: fragment reads of 16 rows start in different banks
constexpr int kPartFloats = 32 * 33;     // a wave's sums

struct __attribute__((packed, aligned(4))) Floats4 {
    Bytes16 v;
};
__device__ __forceinline__ Bytes16 Load4(const float* p) { return reinterpret_cast<const Floats4*>(p)->v; }

// The run of 4 terms from k on of a row of K.  Of a row of 4 and more, what lies beyond it comes from in front of the run instead (16 bytes inside the
// row, wherever k is); KeepRun drops that.  Shorter rows are read one by one.
__device__ __forceinline__ int RunStart(int k, int K) { return K >= 4 ? min(k, K - 4) : k; }
// The runs from k on of four rows.
__device__ __forceinline__ void LoadRuns(const float* const (&row)[4], int k, int K, Bytes16 (&v)[4]) {
    if (K >= 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = Load4(row[j] + RunStart(k, K));
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] = __float_as_uint(row[j][min(k + e, K - 1)]);
}
__device__ __forceinline__ void KeepRun(Bytes16& v, int k, int K) {
    const int at = RunStart(k, K);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (at + e >= k) & (at + e < K) ? v[e] : 0u;
}

// One unit of one row: x and h are the two sides' pre-activations with their biases (Linear(x), Linear(h)).  Returns the new state; `gates`, if not null, is
// where its saved values go, H apart.
template <int MODE, int G>
__device__ __forceinline__ float RunCell(const float (&x)[G], const float (&h)[G], float h_old, float c_old, bool relu, float* gates, int H, float& c_new) {
    auto pre = [&](int g) { return x[g] + h[g]; };
    if constexpr (MODE == kLstm) {
        const float gi = Sigmoid(pre(0)), gf = Sigmoid(pre(1)), gg = tanhf(pre(2)), go = Sigmoid(pre(3));
        c_new = gg * gi + gf * c_old;
        if (gates != nullptr) gates[0] = gi, gates[H] = gf, gates[2 * H] = gg, gates[3 * H] = go;
        return go * tanhf(c_new);
    } else if constexpr (MODE == kGru) {
        const float gr = Sigmoid(pre(0)), gz = Sigmoid(pre(1));
        const float gn = tanhf(x[2] + gr * h[2]);
        if (gates != nullptr) gates[0] = gr, gates[H] = gz, gates[2 * H] = gn, gates[3 * H] = h[2];
        return (1.0f - gz) * gn + gz * h_old;
    } else {
        const float h_new = relu ? fmaxf(pre(0), 0.0f) : tanhf(pre(0));
        if (gates != nullptr) *gates = h_new;
        return h_new;
    }
}

// One step of one layer-direction.  Matrices are dense [units][columns], vectors dense.
struct StepJob {
    const float* x;  // [bt] rows of the layer's input; null: its projection is in xw
    int64_t x_stride;
    int in;
    int bt;
    int prev_rows;       // the state before the step of rows below it is in h_prev (the outputs of the step before), of the others in h0
    const float* h_prev;
    int64_t h_prev_stride;
    const float* h0;     // [B][H]
    const float* xw;     // [bt][G*H]
    const float* wx[4];  // per gate
    const float* wh[4];
    const float* bx[4];
    const float* bh[4];
    float* y;            // [bt] output rows
    int64_t y_stride;
    float* hy;           // the state after the last step of each row: rows < bt are written
    int64_t hy_row, hy_col;
    float* cy;           // (LSTM) the same, and the state before the step
    int64_t cy_row, cy_col;
    float* gates;        // reserve, this step's rows [bt][GR*H]; null: inference
    float* hprev;        // reserve [bt][H]
    float* cprev;        // reserve [bt][H] (LSTM)
};

struct StepArgs {
    int relu;
    int H;
    StepJob job[kMaxJobs];
};

// The products x . Wx^T and h . Wh^T of a step and the cells in one launch.  A workgroup owns 32 rows and the gates of 8 (RNN: 32) units, so that the
// sums of its eight waves, which split the reduction, meet in LDS and the cells run on them: gate pre-activations never reach memory.  GRU keeps
// the sums of the two sides apart, as its last gate needs them (and takes the columns of a fourth gate, which nobody reads).
// A wave reads whole lines (8 lanes to a row) two chunks ahead and turns them round in LDS of its own: read straight into the MFMA layout, 32 rows to
// an instruction, the loads alone took 14 us a step at [20,1300] . [1300,2600], 64 clocks an instruction.
// Bound by latency (launch, first loads, the waves' sums): a launch advances every layer-direction that can go (blockIdx.y), and whatever the cells
// read is loaded ahead of the products.  Two layers of 650 LSTM units, 20 rows, 35 steps: 70 launches
// each of a product (4.9 us) and of cells (4.5) -> 36 of 13.4, x's products (88 us) and the packing of the weights included.
template <int MODE>
__global__ __launch_bounds__(64 * kStepWaves) void RnnStepKernel(StepArgs p) {
    constexpr int G = MODE == kLstm ? 4 : (MODE == kGru ? 3 : 1);
    constexpr int C = G == 1 ? 1 : 4;  // columns of a unit
    constexpr int UNITS = 32 / C;
    constexpr int SIDES = MODE == kGru ? 2 : 1;
    constexpr int CELLS = 32 * UNITS / (64 * kStepWaves) > 1 ? 32 * UNITS / (64 * kStepWaves) : 1;  // of a thread
    static_assert(SIDES * kPartFloats * 4 <= 2 * 32 * kPitch, "the sums fit the staging areas");
    __shared__ __align__(16) char lds[kStepWaves * 2 * 32 * kPitch];
    const StepJob& args = p.job[blockIdx.y];
    const float* const x_rows = args.x;
    const float* const xw_rows = args.xw;
    const float* const h_prev = args.h_prev;
    const float* const h0 = args.h0;
    const int64_t x_stride = args.x_stride, h_prev_stride = args.h_prev_stride, y_stride = args.y_stride;
    const int bt = args.bt, prev_rows = args.prev_rows, in = x_rows != nullptr ? args.in : 0;
    float *const y = args.y, *const hy = args.hy, *const gates = args.gates, *const hprev = args.hprev;
    const int64_t hy_row = args.hy_row, hy_col = args.hy_col;
    float* const cy = MODE == kLstm ? args.cy : nullptr;
    float* const cprev = MODE == kLstm ? args.cprev : nullptr;
    const int64_t cy_row = MODE == kLstm ? args.cy_row : 0, cy_col = MODE == kLstm ? args.cy_col : 0;
    const float *const wx0 = args.wx[0], *const wx1 = args.wx[G > 1], *const wx2 = args.wx[G > 2 ? 2 : 0], *const wx3 = args.wx[G > 3 ? 3 : 0];
    const float *const wh0 = args.wh[0], *const wh1 = args.wh[G > 1], *const wh2 = args.wh[G > 2 ? 2 : 0], *const wh3 = args.wh[G > 3 ? 3 : 0];
    const float *const bx0 = args.bx[0], *const bx1 = args.bx[G > 1], *const bx2 = args.bx[G > 2 ? 2 : 0], *const bx3 = args.bx[G > 3 ? 3 : 0];
    const float *const bh0 = args.bh[0], *const bh1 = args.bh[G > 1], *const bh2 = args.bh[G > 2 ? 2 : 0], *const bh3 = args.bh[G > 3 ? 3 : 0];
    Pin(x_rows, xw_rows, h_prev, h0, x_stride, h_prev_stride, y_stride, bt, prev_rows, in, y, hy, gates, hprev, hy_row, hy_col, cy, cprev, cy_row, cy_col);
    Pin(wx0, wx1, wx2, wx3, wh0, wh1, wh2, wh3, bx0, bx1, bx2, bx3, bh0, bh1, bh2, bh3);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, half = lane >> 5;
    const int H = p.H;
    const int tiles_m = (bt + 31) / 32, tiles = tiles_m * ((H + UNITS - 1) / UNITS);
    if (static_cast<int>(blockIdx.x) >= tiles) return;
    int tm, tn;
    SmallDotTile(tiles, blockIdx.x, tiles_m, tm, tn);

    // what this thread's cells read
    float xw[CELLS][G], b_x[CELLS][G], b_h[CELLS][G], h_old[CELLS], c_old[CELLS];
    auto cell_at = [&](int i, int& r, int& u) {
        const int e = tid + i * 64 * kStepWaves;
        r = tm * 32 + e / UNITS, u = tn * UNITS + e % UNITS;
        return e < 32 * UNITS && r < bt && u < H;
    };
    auto state_row = [&](int r) -> const float* { return r < prev_rows ? h_prev + r * h_prev_stride : h0 + static_cast<int64_t>(r) * H; };
#pragma unroll
    for (int i = 0; i < CELLS; ++i) {
        int r, u;
        if (!cell_at(i, r, u)) continue;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            xw[i][g] = xw_rows != nullptr ? xw_rows[(static_cast<int64_t>(r) * G + g) * H + u] : 0.f;
            b_x[i][g] = (g == 0 ? bx0 : (g == 1 ? bx1 : (g == 2 ? bx2 : bx3)))[u];
            b_h[i][g] = (g == 0 ? bh0 : (g == 1 ? bh1 : (g == 2 ? bh2 : bh3)))[u];
        }
        h_old[i] = state_row(r)[u];
        if constexpr (MODE == kLstm) c_old[i] = cy[r * cy_row + u * cy_col];
    }

    // ---- products: this lane's piece (4 k) of every eighth row of x and h and of the matrices' rows that are the columns (rows and columns beyond the
    // problem repeat the last one: nobody reads what comes of them) ----
    const int piece = (lane & 7) * 4, eighth = lane >> 3;
    const int gate = eighth % C;  // of this lane's columns j * 8 + eighth
    const float* const w_x = gate == 0 ? wx0 : (gate == 1 ? wx1 : (gate == 2 ? wx2 : wx3));
    const float* const w_h = gate == 0 ? wh0 : (gate == 1 ? wh1 : (gate == 2 ? wh2 : wh3));
    const float *x_row[4], *h_row[4], *wx_row[4], *wh_row[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int row = min(tm * 32 + j * 8 + eighth, bt - 1);
        const int64_t unit = min(tn * UNITS + (j * 8 + eighth) / C, H - 1);
        x_row[j] = x_rows + row * x_stride;
        h_row[j] = state_row(row);
        wx_row[j] = w_x + unit * in;
        wh_row[j] = w_h + unit * H;
    }
    const int chunks_x = (in + kChunk - 1) / kChunk, chunks = chunks_x + (H + kChunk - 1) / kChunk;
    const int per_wave = (chunks + kStepWaves - 1) / kStepWaves;
    const int begin = min(chunks, wave * per_wave), n = min(chunks, begin + per_wave) - begin;
    float16_t acc[SIDES];
#pragma unroll
    for (int s = 0; s < SIDES; ++s)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[s][v] = 0.f;
    Bytes16 av[2][4], bv[2][4];
    auto load = [&](int st, int c) {
        const int i = begin + c;
        if (i < chunks_x) {
            LoadRuns(x_row, i * kChunk + piece, in, av[st]);
            LoadRuns(wx_row, i * kChunk + piece, in, bv[st]);
        } else {
            LoadRuns(h_row, (i - chunks_x) * kChunk + piece, H, av[st]);
            LoadRuns(wh_row, (i - chunks_x) * kChunk + piece, H, bv[st]);
        }
    };
    char* const stage = lds + wave * 2 * 32 * kPitch;
    auto multiply = [&](int st, int c) {
        const int i = begin + c;
        const bool x = i < chunks_x;
        const int k = (x ? i : i - chunks_x) * kChunk, K = x ? in : H;
        if (k + kChunk > K) {
#pragma unroll
            for (int j = 0; j < 4; ++j) KeepRun(av[st][j], k + piece, K), KeepRun(bv[st][j], k + piece, K);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            *reinterpret_cast<Bytes16*>(stage + (j * 8 + eighth) * kPitch + piece * 4) = av[st][j];
            *reinterpret_cast<Bytes16*>(stage + (32 + j * 8 + eighth) * kPitch + piece * 4) = bv[st][j];
        }
        if (c + 2 < n) load(st, c + 2);
        __builtin_amdgcn_wave_barrier();
        Bytes16 fa[4], fb[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            fa[q] = *reinterpret_cast<const Bytes16*>(stage + lr * kPitch + (2 * q + half) * 16);
            fb[q] = *reinterpret_cast<const Bytes16*>(stage + (32 + lr) * kPitch + (2 * q + half) * 16);
        }
        if (SIDES == 1 || x) {
#pragma unroll
            for (int q = 0; q < 4; ++q) MfmaTile<float>(fa[q], fb[q], acc[0]);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) MfmaTile<float>(fa[q], fb[q], acc[SIDES - 1]);
        }
        __builtin_amdgcn_wave_barrier();
    };
    if (n > 0) load(0, 0);
    if (n > 1) load(1, 1);
    for (int c = 0; c < n; c += 2) {
        multiply(0, c);
        if (c + 1 < n) multiply(1, c + 1);
    }
    __syncthreads();  // the staging areas become the sums
    float* const part = reinterpret_cast<float*>(lds);
    // lane holds column lr, rows 8 * (v / 4) + 4 * half + v % 4
#pragma unroll
    for (int s = 0; s < SIDES; ++s)
#pragma unroll
        for (int v = 0; v < 16; ++v) part[(s * kStepWaves + wave) * kPartFloats + (8 * (v / 4) + 4 * half + v % 4) * 33 + lr] = acc[s][v];
    __syncthreads();

#pragma unroll
    for (int i = 0; i < CELLS; ++i) {
        int r, u;
        if (!cell_at(i, r, u)) continue;
        const int at = (r - tm * 32) * 33 + (u - tn * UNITS) * C;
        float sum[SIDES][G];
#pragma unroll
        for (int s = 0; s < SIDES; ++s)
#pragma unroll
            for (int g = 0; g < G; ++g) {
                sum[s][g] = 0.f;
#pragma unroll
                for (int w = 0; w < kStepWaves; ++w) sum[s][g] += part[(s * kStepWaves + w) * kPartFloats + at + g];
            }
        const int64_t idx = static_cast<int64_t>(r) * H + u;
        float from_x[G], from_h[G], c_new = 0.f;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            from_x[g] = (MODE == kGru ? xw[i][g] + sum[0][g] : xw[i][g]) + b_x[i][g];
            from_h[g] = sum[SIDES - 1][g] + b_h[i][g];
        }
        float* const saved = gates != nullptr ? gates + (static_cast<int64_t>(r) * (G == 1 ? 1 : 4) * H + u) : nullptr;
        const float h_new = RunCell<MODE, G>(from_x, from_h, h_old[i], c_old[i], p.relu != 0, saved, H, c_new);
        if constexpr (MODE == kLstm) {
            cy[r * cy_row + u * cy_col] = c_new;
            if (gates != nullptr) cprev[idx] = c_old[i];
        }
        if (gates != nullptr) hprev[idx] = h_old[i];
        hy[r * hy_row + u * hy_col] = h_new;
        y[r * y_stride + u] = h_new;
    }
}

// The cells of a step whose products are in memory, [bt][G*H]; states [B][H] are updated in place.
struct CellJob {
    int bt;
    const float* xw;
    const float* hw;
    const float* bx[4];
    const float* bh[4];
    float* h;
    float* c;  // (LSTM)
    int64_t c_row, c_col;
    float* y;
    int64_t y_stride;
    float* gates;  // as in StepJob
    float* hprev;
    float* cprev;
};

struct CellArgs {
    int relu;
    int H;
    CellJob job[2];
};

template <int MODE>
__global__ __launch_bounds__(256) void RnnCellKernel(CellArgs p) {
    constexpr int G = MODE == kLstm ? 4 : (MODE == kGru ? 3 : 1);
    const CellJob& j = p.job[blockIdx.y];
    const int H = p.H, total = j.bt * H;
    for (int idx = blockIdx.x * 256 + threadIdx.x; idx < total; idx += gridDim.x * 256) {
        const int r = idx / H, u = idx - r * H;
        float from_x[G], from_h[G], c_old = 0.f, c_new = 0.f;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int64_t at = (static_cast<int64_t>(r) * G + g) * H + u;
            from_x[g] = j.xw[at] + j.bx[g][u];
            from_h[g] = j.hw[at] + j.bh[g][u];
        }
        const float h_old = j.h[idx];
        if constexpr (MODE == kLstm) c_old = j.c[r * j.c_row + u * j.c_col];
        float* const saved = j.gates != nullptr ? j.gates + (static_cast<int64_t>(r) * (G == 1 ? 1 : 4) * H + u) : nullptr;
        const float h_new = RunCell<MODE, G>(from_x, from_h, h_old, c_old, p.relu != 0, saved, H, c_new);
        if constexpr (MODE == kLstm) j.c[r * j.c_row + u * j.c_col] = c_new;
        if (j.gates != nullptr) {
            j.hprev[idx] = h_old;
            if constexpr (MODE == kLstm) j.cprev[idx] = c_old;
        }
        j.h[idx] = h_new;
        j.y[static_cast<int64_t>(r) * j.y_stride + u] = h_new;
    }
}

struct CellGradJob {
    int bt;
    const float* dy;     // this step's rows of the gradient of the layer's output, this direction's columns: dy_splits parts dy_part floats apart
    int64_t dy_stride;
    int dy_splits;
    int64_t dy_part;
    float* dh;           // [B][H]: the part of the gradient of the state after the step that did not pass through Wh in the step behind it;
                         // out, the same for the step before (GRU: dh * z, else 0)
    const float* parts;  // [splits][part_rows][H]: the other part, dGh . Wh of the step behind, in parts of its reduction
    int splits, part_rows;
    float* dc;           // [B][H] (LSTM), updated in place
    const float* gates;
    const float* hprev;
    const float* cprev;
    float* dgx;          // [bt][G*H]: gradient of x . Wx^T + bx
    float* dgh;          // [bt][G*H]: gradient of h . Wh^T + bh (the same array as dgx unless GRU)
};

struct CellGradArgs {
    int relu;
    int H;
    CellGradJob job[kMaxJobs];
};

// sum of p[s * stride], s < splits, in that order
__device__ __forceinline__ float SumParts(const float* p, int splits, int64_t stride) {
    float sum = 0.f;
#pragma unroll 8
    for (int s = 0; s < splits; ++s) sum += p[s * stride];
    return sum;
}

// Rows from bt to part_rows, which the step does not hold, only take in their parts.  blockIdx.y: the layer-direction.
template <int MODE>
__global__ __launch_bounds__(256) void RnnCellGradKernel(CellGradArgs p) {
    const CellGradJob& args = p.job[blockIdx.y];
    const int bt = args.bt, splits = args.splits, part_rows = args.part_rows, dy_splits = args.dy_splits;
    const int64_t dy_stride = args.dy_stride, dy_part = args.dy_part;
    const float *const dy = args.dy, *const parts = args.parts, *const gates = args.gates, *const hprev = args.hprev, *const cprev = args.cprev;
    float *const dh_state = args.dh, *const dc_state = args.dc, *const dgx = args.dgx, *const dgh = args.dgh;
    Pin(bt, splits, part_rows, dy_splits, dy_stride, dy_part, dy, parts, gates, hprev, cprev, dh_state, dc_state, dgx, dgh);
    const int H = p.H;
    const int total = max(bt, part_rows) * H;
    for (int idx = blockIdx.x * 256 + threadIdx.x; idx < total; idx += gridDim.x * 256) {
        const int r = idx / H, u = idx - r * H;
        float* dhs = dh_state + idx;
        float after = *dhs;
        if (r < part_rows) after += SumParts(parts + idx, splits, static_cast<int64_t>(part_rows) * H);
        if (r >= bt) {
            *dhs = after;
            continue;
        }
        const float dh = after + SumParts(dy + r * dy_stride + u, dy_splits, dy_part);
        if constexpr (MODE == kLstm) {
            const float* q = gates + static_cast<int64_t>(r) * 4 * H + u;
            const float gi = q[0], gf = q[H], gg = q[2 * H], go = q[3 * H];
            const float c_old = cprev[idx];
            const float tc = tanhf(gg * gi + gf * c_old);
            float* dcs = dc_state + idx;
            const float dc = *dcs + dh * go * (1.0f - tc * tc);
            float* g = dgx + static_cast<int64_t>(r) * 4 * H + u;
            g[0] = dc * gg * gi * (1.0f - gi);
            g[H] = dc * c_old * gf * (1.0f - gf);
            g[2 * H] = dc * gi * (1.0f - gg * gg);
            g[3 * H] = dh * tc * go * (1.0f - go);
            *dcs = dc * gf;
            *dhs = 0.0f;
        } else if constexpr (MODE == kGru) {
            const float* q = gates + static_cast<int64_t>(r) * 4 * H + u;
            const float gr = q[0], gz = q[H], gn = q[2 * H], hh = q[3 * H];
            const float h_old = hprev[idx];
            const float dn_pre = dh * (1.0f - gz) * (1.0f - gn * gn);
            const float dz_pre = dh * (h_old - gn) * gz * (1.0f - gz);
            const float dr_pre = dn_pre * hh * gr * (1.0f - gr);
            float* gx = dgx + static_cast<int64_t>(r) * 3 * H + u;
            float* gh = dgh + static_cast<int64_t>(r) * 3 * H + u;
            gx[0] = dr_pre, gx[H] = dz_pre, gx[2 * H] = dn_pre;
            gh[0] = dr_pre, gh[H] = dz_pre, gh[2 * H] = dn_pre * gr;
            *dhs = dh * gz;
        } else {
            const float h_new = gates[idx];
            dgx[idx] = p.relu ? (h_new > 0.0f ? dh : 0.0f) : dh * (1.0f - h_new * h_new);
            *dhs = 0.0f;
        }
    }
}

// What a step's gate gradients mean for the state before it and, where the layer below runs a step behind, for the layer's input.
struct BackJob {
    int bt;
    const float* dgh;    // [bt][G*H]
    const float* dgx;
    const float* wh[4];  // per gate [H][H]
    const float* wx[4];  // per gate [H][in]
    int in;              // 0: the input's gradient is not wanted
    float* dh_parts;     // [splits][bt][H]
    float* dx_parts;     // [splits][bt][in]
};

struct BackArgs {
    int G, H;
    int subs;  // parts of a gate's reduction; splits = G * subs
    BackJob job[kMaxJobs];
};

// The products dGh . Wh and dGx . Wx of a step, in parts of the reduction which the cell kernel adds up: a workgroup owns 32 rows, 32 columns and a
// part of one gate's units, its eight waves split that.  The rows come as whole lines, turned round in LDS; the matrices, whose rows are k, element by
// element with the columns across the lanes: whole lines too, already in the MFMA layout.  Bound by latency like the forward step.
__global__ __launch_bounds__(64 * kStepWaves) void RnnBackKernel(BackArgs p) {
    __shared__ __align__(16) char lds[kStepWaves * 32 * kPitch];
    const BackJob& args = p.job[blockIdx.y];
    const int bt = args.bt, in = args.in;
    const float *const dgh = args.dgh, *const dgx = args.dgx;
    const float *const wh0 = args.wh[0], *const wh1 = args.wh[1], *const wh2 = args.wh[2], *const wh3 = args.wh[3];
    const float *const wx0 = args.wx[0], *const wx1 = args.wx[1], *const wx2 = args.wx[2], *const wx3 = args.wx[3];
    float *const dh_parts = args.dh_parts, *const dx_parts = args.dx_parts;
    Pin(bt, in, dgh, dgx, wh0, wh1, wh2, wh3, wx0, wx1, wx2, wx3, dh_parts, dx_parts);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, half = lane >> 5;
    const int H = p.H, splits = p.G * p.subs;
    const int tiles_m = (bt + 31) / 32, tiles_h = (H + 31) / 32, tiles_n = tiles_h + (in + 31) / 32;
    const int tiles = tiles_m * tiles_n;
    if (static_cast<int>(blockIdx.x) >= tiles * splits) return;
    const int split = blockIdx.x / tiles;
    int tm, tn;
    SmallDotTile(tiles, blockIdx.x - split * tiles, tiles_m, tm, tn);
    const bool state = tn < tiles_h;
    const int N = state ? H : in;
    const int n0 = (state ? tn : tn - tiles_h) * 32;
    const int gate = split / p.subs, sub = split - gate * p.subs;
    const float* const w_h = gate == 0 ? wh0 : (gate == 1 ? wh1 : (gate == 2 ? wh2 : wh3));
    const float* const w_x = gate == 0 ? wx0 : (gate == 1 ? wx1 : (gate == 2 ? wx2 : wx3));
    const int piece = (lane & 7) * 4, eighth = lane >> 3, col = min(n0 + lr, N - 1);
    const float* a[4];  // every eighth row
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j] = (state ? dgh : dgx) + (static_cast<int64_t>(min(tm * 32 + j * 8 + eighth, bt - 1)) * p.G + gate) * H;
    const float* const b = (state ? w_h : w_x) + col;

    const int chunks = (H + kChunk - 1) / kChunk, per_sub = (chunks + p.subs - 1) / p.subs;
    const int sub_begin = min(chunks, sub * per_sub), sub_end = min(chunks, sub_begin + per_sub);
    const int per_wave = (sub_end - sub_begin + kStepWaves - 1) / kStepWaves;
    const int begin = min(sub_end, sub_begin + wave * per_wave), end = min(sub_end, begin + per_wave);
    float16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    char* const stage = lds + wave * 32 * kPitch;
    Bytes16 av[2][4], bv[2][4];
    auto load = [&](int st, int c) {
        const int k = c * kChunk;
        LoadRuns(a, k + piece, H, av[st]);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) bv[st][q][e] = __float_as_uint(b[static_cast<int64_t>(min(k + (2 * q + half) * 4 + e, H - 1)) * N]);
    };
    auto multiply = [&](int st, int c) {
        const int k = c * kChunk;
        if (k + kChunk > H) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                KeepRun(av[st][j], k + piece, H);
                // to where the matrices' elements are
                Bytes16 v = av[st][j];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int shift = k + piece - RunStart(k + piece, H);  // the run was read that much too early
                    av[st][j][e] = e + shift < 4 ? (shift == 0 ? v[e] : (shift == 1 ? v[(e + 1) & 3] : (shift == 2 ? v[(e + 2) & 3] : v[(e + 3) & 3]))) : 0u;
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) bv[st][q][e] = k + (2 * q + half) * 4 + e < H ? bv[st][q][e] : 0u;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) *reinterpret_cast<Bytes16*>(stage + (j * 8 + eighth) * kPitch + piece * 4) = av[st][j];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const Bytes16 fa = *reinterpret_cast<const Bytes16*>(stage + lr * kPitch + (2 * q + half) * 16);
            MfmaTile<float>(fa, bv[st][q], acc);
        }
        if (c + 2 < end) load(st, c + 2);
        __builtin_amdgcn_wave_barrier();
    };
    if (begin < end) load(0, begin);
    if (begin + 1 < end) load(1, begin + 1);
    for (int c = begin; c < end; c += 2) {
        multiply(0, c);
        if (c + 1 < end) multiply(1, c + 1);
    }
    __syncthreads();  // the staging areas become the sums
    float* const part = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int v = 0; v < 16; ++v) part[wave * kPartFloats + (8 * (v / 4) + 4 * half + v % 4) * 33 + lr] = acc[v];
    __syncthreads();
    float* const out = (state ? dh_parts : dx_parts) + static_cast<int64_t>(split) * bt * N;
    for (int e = tid; e < 32 * 32; e += 64 * kStepWaves) {
        const int row = e >> 5, c = e & 31;
        if (tm * 32 + row >= bt || n0 + c >= N) continue;
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < kStepWaves; ++w) s += part[w * kPartFloats + row * 33 + c];
        out[static_cast<int64_t>(tm * 32 + row) * N + n0 + c] = s;
    }
}

// f<mode> for the mode of a call
template <typename F>
void VisitMode(int mode, F&& f) {
    if (mode == kLstm) f(std::integral_constant<int, kLstm>{});
    else if (mode == kGru) f(std::integral_constant<int, kGru>{});
    else f(std::integral_constant<int, kRnn>{});
}

size_t Round256(size_t v) { return (v + 255) / 256 * 256; }

void CheckStatus(int status) {
    if (status != HIPCX_OK) throw Error(status, hipcx_last_error());
}

hipcx_array Matrix(const void* data, int64_t rows, int64_t cols, int64_t row_stride, int64_t col_stride = 1) {
    hipcx_array a{};
    a.data = const_cast<void*>(data);
    a.dtype = HIPCX_FLOAT32;
    a.ndim = 2;
    a.shape[0] = rows, a.shape[1] = cols;
    a.strides[0] = row_stride * 4, a.strides[1] = col_stride * 4;
    return a;
}

hipcx_array Vector(const void* data, int64_t n, int64_t stride = 1) {
    hipcx_array a{};
    a.data = const_cast<void*>(data);
    a.dtype = HIPCX_FLOAT32;
    a.ndim = 1;
    a.shape[0] = n;
    a.strides[0] = stride * 4;
    return a;
}

// Shapes of a call and the layout of its workspace and reserve.  Offsets are bytes.
struct RnnPlan {
    int L = 0, D = 1, T = 0, mode = 0, G = 1, GR = 1;
    int64_t B = 0, H = 0, I = 0, rows = 0, max_in = 0;
    std::vector<int64_t> row_start, bt;
    // reserve (forward writes, backward reads): per layer-direction the gate activations and the states before each step; per
    // layer below the top its output rows
    std::vector<size_t> r_gates, r_hprev, r_cprev, r_y;
    size_t reserve_total = 0;
    int64_t In(int layer) const { return layer == 0 ? I : D * H; }
};

RnnPlan MakePlan(int n_layers, int bidirectional, int mode, const hipcx_array* hx, const hipcx_array* const* xs, int n_steps) {
    HIPCX_REQUIRE(mode == kGru || mode == kLstm || mode == kRnn, HIPCX_CHAINERX_ERROR, "n_step_rnn: mode must be 0 (GRU), 1 (LSTM) or 2 (RNN)");
    HIPCX_REQUIRE(n_layers >= 1 && n_steps >= 1, HIPCX_DIMENSION_ERROR, "n_step_rnn: at least one layer and one time step are required");
    HIPCX_REQUIRE(xs != nullptr, HIPCX_CHAINERX_ERROR, "xs is null");
    ValidateArray(hx, "hx");
    RnnPlan pl;
    pl.L = n_layers, pl.D = bidirectional ? 2 : 1, pl.T = n_steps, pl.mode = mode;
    pl.G = NumGates(mode), pl.GR = ReserveGates(mode);
    HIPCX_REQUIRE(hx->ndim == 3 && hx->shape[0] == n_layers * pl.D, HIPCX_DIMENSION_ERROR,
                  "hx must have the shape [n_layers * directions, batch, units], got " + ShapeStr(hx));
    HIPCX_REQUIRE(hx->dtype == HIPCX_FLOAT32, HIPCX_NOT_IMPLEMENTED_ERROR, "hip n_step_rnn: float32 only (compose the routine for other dtypes)");
    pl.B = hx->shape[1], pl.H = hx->shape[2];
    HIPCX_REQUIRE(pl.B > 0 && pl.H > 0 && pl.B < (1 << 24) && pl.H < (1 << 24), HIPCX_NOT_IMPLEMENTED_ERROR, "hip n_step_rnn: empty or oversized state");
    for (int t = 0; t < n_steps; ++t) {
        ValidateArray(xs[t], "xs[t]");
        HIPCX_REQUIRE(xs[t]->ndim == 2, HIPCX_DIMENSION_ERROR, "every xs[t] must be a matrix");
        HIPCX_REQUIRE(xs[t]->dtype == HIPCX_FLOAT32, HIPCX_NOT_IMPLEMENTED_ERROR, "hip n_step_rnn: float32 only");
        if (t == 0) pl.I = xs[0]->shape[1];
        HIPCX_REQUIRE(xs[t]->shape[1] == pl.I && pl.I > 0 && pl.I < (1 << 24), HIPCX_DIMENSION_ERROR, "every xs[t] must have the same number of columns");
        HIPCX_REQUIRE(xs[t]->shape[0] <= pl.B, HIPCX_DIMENSION_ERROR, "The batch size of x must be equal to or less than the size of state");
        HIPCX_REQUIRE(xs[t]->shape[0] > 0, HIPCX_NOT_IMPLEMENTED_ERROR, "hip n_step_rnn: empty time step");
        pl.row_start.push_back(pl.rows);
        pl.bt.push_back(xs[t]->shape[0]);
        pl.rows += xs[t]->shape[0];
    }
    HIPCX_REQUIRE(pl.rows * std::max<int64_t>(pl.I, 4 * pl.D * pl.H) < (int64_t{1} << 31), HIPCX_NOT_IMPLEMENTED_ERROR, "hip n_step_rnn: sequence batch too large");
    pl.max_in = std::max(pl.I, pl.D * pl.H);
    size_t off = 0;
    for (int idx = 0; idx < pl.L * pl.D; ++idx) {
        pl.r_gates.push_back(off);
        off += Round256(static_cast<size_t>(pl.rows * pl.GR * pl.H) * 4);
        pl.r_hprev.push_back(off);
        off += Round256(static_cast<size_t>(pl.rows * pl.H) * 4);
        pl.r_cprev.push_back(off);
        if (mode == kLstm) off += Round256(static_cast<size_t>(pl.rows * pl.H) * 4);
    }
    for (int l = 0; l + 1 < pl.L; ++l) {
        pl.r_y.push_back(off);
        off += Round256(static_cast<size_t>(pl.rows * pl.D * pl.H) * 4);
    }
    pl.reserve_total = off;
    return pl;
}

// Hands out pieces of the workspace and runs the library calls of a pass.  In a dry run (base == nullptr) nothing is launched: the
// pieces get addresses relative to an aligned dummy base and the scratch need of every product / sum is recorded, which is how
// the workspace size of a pass is computed from the same code that later runs it.
class Pass {
public:
    Pass(void* base, size_t bytes, void* stream) : base_(static_cast<char*>(base)), bytes_(bytes), stream_(stream), dry_(base == nullptr) {
        if (dry_) base_ = reinterpret_cast<char*>(uintptr_t{1} << 20);
    }
    bool dry() const { return dry_; }
    hipStream_t hip_stream() const { return AsStream(stream_); }
    float* Take(int64_t floats) {
        float* p = reinterpret_cast<float*>(base_ + used_);
        used_ += Round256(static_cast<size_t>(floats) * 4);
        return p;
    }
    // everything after the pieces is scratch for the library calls; call once all pieces are taken, before anything is launched
    void StartScratch() {
        scratch_off_ = used_;
        CheckFits();
    }
    size_t Need() const { return scratch_off_ + scratch_need_; }
    void CheckFits() const {
        HIPCX_REQUIRE(dry_ || Need() <= bytes_, HIPCX_CHAINERX_ERROR, "n_step_rnn workspace too small: need " + std::to_string(Need()) + " bytes");
    }
    void Dot(const hipcx_array& a, const hipcx_array& b, const hipcx_array& out) {
        const size_t need = hipcx_dot_workspace_size(&a, &b, &out);
        if (dry_) {
            scratch_need_ = std::max(scratch_need_, Round256(need));
            return;
        }
        HIPCX_REQUIRE(scratch_off_ + need <= bytes_, HIPCX_CHAINERX_ERROR, "n_step_rnn workspace too small for a matrix product");
        CheckStatus(hipcx_dot(&a, &b, &out, base_ + scratch_off_, bytes_ - scratch_off_, stream_));
    }
    void SumRows(const hipcx_array& a, const hipcx_array& out) {
        const int8_t axis = 0;
        const size_t need = hipcx_reduce_workspace_size(&a, &axis, 1, &out);
        if (dry_) {
            scratch_need_ = std::max(scratch_need_, Round256(need));
            return;
        }
        HIPCX_REQUIRE(scratch_off_ + need <= bytes_, HIPCX_CHAINERX_ERROR, "n_step_rnn workspace too small for a sum");
        CheckStatus(hipcx_sum(&a, &axis, 1, &out, base_ + scratch_off_, bytes_ - scratch_off_, stream_));
    }
    // outs[i] = a_i . b for left operands `distance` elements apart
    void DotEach(const hipcx_array& a0, int64_t distance, const hipcx_array& b, const hipcx_array* const* outs, int n) {
        if (!dry_ && DotSeveral(&a0, distance, &b, outs, n, hip_stream())) return;
        hipcx_array a = a0;
        for (int i = 0; i < n; ++i) {
            Dot(a, b, *outs[i]);
            a.data = static_cast<float*>(a.data) + distance;
        }
    }
    // Copies run together, at the next FlushCopies()
    void Copy(const hipcx_array& a, const hipcx_array& out) {
        copies_.push_back(a);
        copies_.push_back(out);
    }
    void FlushCopies() {
        if (copies_.empty()) return;
        std::vector<const hipcx_array*> from, to;
        for (size_t i = 0; i < copies_.size(); i += 2) {
            from.push_back(&copies_[i]);
            to.push_back(&copies_[i + 1]);
        }
        if (!dry_) CheckStatus(hipcx_copy_many(from.data(), to.data(), static_cast<int>(from.size()), stream_));
        copies_.clear();
    }
    void Add(const hipcx_array& a, const hipcx_array& b, const hipcx_array& out) {
        if (!dry_) CheckStatus(hipcx_add(&a, &b, &out, stream_));
    }
    void Zero(const hipcx_array& out) {
        hipcx_scalar zero{};
        zero.kind = HIPCX_KIND_INT;
        if (!dry_) CheckStatus(hipcx_fill(&out, zero, stream_));
    }

private:
    char* base_;
    size_t bytes_;
    void* stream_;
    bool dry_;
    size_t used_ = 0, scratch_off_ = 0, scratch_need_ = 0;
    std::vector<hipcx_array> copies_;
};

// The matrices of a layer-direction's x side (first = 0) or h side (first = G) stacked gate-major into [G*H][columns]: rows [g*H, (g+1)*H) are
// ws[idx][first + g].
float* PackWeights(Pass& pass, const RnnPlan& pl, const hipcx_array* const* ws, int idx, int first) {
    const int64_t columns = first == 0 ? pl.In(idx / pl.D) : pl.H;
    float* const packed = pass.Take(pl.G * pl.H * columns);
    if (pass.dry()) return packed;
    for (int g = 0; g < pl.G; ++g) pass.Copy(*ws[idx * 2 * pl.G + first + g], Matrix(packed + g * pl.H * columns, pl.H, columns, columns));
    return packed;
}

// The bytes that an array spans.
struct Span {
    uintptr_t begin, end;
    const hipcx_array* array;
};
Span SpanOf(const hipcx_array* a) {
    Span s{reinterpret_cast<uintptr_t>(a->data), reinterpret_cast<uintptr_t>(a->data) + 4, a};
    for (int i = 0; i < a->ndim; ++i) {
        const int64_t reach = (a->shape[i] - 1) * a->strides[i];
        (reach < 0 ? s.begin : s.end) += static_cast<uintptr_t>(reach);
    }
    return s;
}

// Whether two arrays may share memory.  Matrices of dense rows with the same distance, as the steps of one batch-major array are, interleave.
bool MayShare(const Span& a, const Span& b) {
    if (a.end <= b.begin || b.end <= a.begin) return false;
    const hipcx_array &x = *a.array, &y = *b.array;
    if (x.ndim != 2 || y.ndim != 2 || x.strides[1] != 4 || y.strides[1] != 4 || x.strides[0] != y.strides[0] || x.strides[0] <= 0) return true;
    const int64_t pitch = x.strides[0];
    int64_t r = static_cast<int64_t>(b.begin - a.begin) % pitch;
    if (r < 0) r += pitch;
    return r < x.shape[1] * 4 || pitch - r < y.shape[1] * 4;
}

// Whether any of `outs` may share memory with another one of them or with one of `ins`.
bool AnyShared(const std::vector<const hipcx_array*>& outs, const std::vector<const hipcx_array*>& ins) {
    std::vector<Span> to, from;
    for (const hipcx_array* a : outs) to.push_back(SpanOf(a));
    for (const hipcx_array* a : ins) from.push_back(SpanOf(a));
    std::sort(to.begin(), to.end(), [](const Span& a, const Span& b) { return a.begin < b.begin; });
    bool apart = true;  // mostly the spans are disjoint
    for (size_t i = 1; i < to.size(); ++i) apart = apart && to[i - 1].end <= to[i].begin;
    for (size_t i = 0; i < from.size() && apart; ++i) {
        const auto behind = std::lower_bound(to.begin(), to.end(), from[i].end, [](const Span& a, uintptr_t end) { return a.begin < end; });
        apart = behind == to.begin() || std::prev(behind)->end <= from[i].begin;
    }
    if (apart) return false;
    for (size_t i = 0; i < to.size(); ++i) {
        for (size_t j = 0; j < i; ++j) {
            if (MayShare(to[i], to[j])) return true;
        }
        for (const Span& f : from) {
            if (MayShare(to[i], f)) return true;
        }
    }
    return false;
}

// An array's data where it is dense and need not be copied, else of a dense copy (there is always room for one: the caller's strides are not known to a
// dry run).
const float* Dense(Pass& pass, const hipcx_array* a, bool copied = false) {
    int64_t n = 1;
    for (int i = 0; i < a->ndim; ++i) n *= a->shape[i];
    float* const copy = pass.Take(n);
    if (pass.dry() || (!copied && IsContiguous(a))) return static_cast<const float*>(a->data);
    pass.Copy(*a, a->ndim == 1 ? Vector(copy, n) : Matrix(copy, a->shape[0], a->shape[1], a->shape[1]));
    return copy;
}

void CheckParameters(const RnnPlan& pl, const hipcx_array* const* ws, const hipcx_array* const* bs, const char* what) {
    HIPCX_REQUIRE(ws != nullptr && bs != nullptr, HIPCX_CHAINERX_ERROR, std::string(what) + " is null");
    for (int idx = 0; idx < pl.L * pl.D; ++idx) {
        const int64_t in = pl.In(idx / pl.D);
        for (int g = 0; g < 2 * pl.G; ++g) {
            const hipcx_array* w = ws[idx * 2 * pl.G + g];
            const hipcx_array* b = bs[idx * 2 * pl.G + g];
            ValidateArray(w, "ws[i]");
            ValidateArray(b, "bs[i]");
            HIPCX_REQUIRE(w->dtype == HIPCX_FLOAT32 && b->dtype == HIPCX_FLOAT32, HIPCX_NOT_IMPLEMENTED_ERROR, "hip n_step_rnn: float32 only");
            HIPCX_REQUIRE(w->ndim == 2 && w->shape[0] == pl.H && w->shape[1] == (g < pl.G ? in : pl.H), HIPCX_DIMENSION_ERROR,
                          std::string(what) + ": matrix " + std::to_string(g) + " of layer-direction " + std::to_string(idx) + " has the wrong shape " +
                                  ShapeStr(w));
            HIPCX_REQUIRE(b->ndim == 1 && b->shape[0] == pl.H, HIPCX_DIMENSION_ERROR, std::string(what) + ": every bias must have one value per unit");
        }
    }
}

void CheckState(const RnnPlan& pl, const hipcx_array* a, const char* name) {
    ValidateArray(a, name);
    HIPCX_REQUIRE(a->dtype == HIPCX_FLOAT32, HIPCX_NOT_IMPLEMENTED_ERROR, "hip n_step_rnn: float32 only");
    HIPCX_REQUIRE(a->ndim == 3 && a->shape[0] == pl.L * pl.D && a->shape[1] == pl.B && a->shape[2] == pl.H, HIPCX_DIMENSION_ERROR,
                  std::string(name) + " must have hx's shape, got " + ShapeStr(a));
}

hipcx_array StateSlice(const hipcx_array* a, int idx) {  // [B][H] view of a[idx]
    hipcx_array m{};
    m.data = static_cast<char*>(a->data) + idx * a->strides[0];
    m.dtype = HIPCX_FLOAT32;
    m.ndim = 2;
    m.shape[0] = a->shape[1], m.shape[1] = a->shape[2];
    m.strides[0] = a->strides[1], m.strides[1] = a->strides[2];
    return m;
}

void CheckStepArrays(const RnnPlan& pl, const hipcx_array* const* arrays, int64_t cols, const char* name, bool nullable) {
    HIPCX_REQUIRE(arrays != nullptr, HIPCX_CHAINERX_ERROR, std::string(name) + " is null");
    for (int t = 0; t < pl.T; ++t) {
        if (arrays[t] == nullptr && nullable) continue;
        ValidateArray(arrays[t], name);
        HIPCX_REQUIRE(arrays[t]->dtype == HIPCX_FLOAT32, HIPCX_NOT_IMPLEMENTED_ERROR, "hip n_step_rnn: float32 only");
        HIPCX_REQUIRE(arrays[t]->ndim == 2 && arrays[t]->shape[0] == pl.bt[t] && arrays[t]->shape[1] == cols, HIPCX_DIMENSION_ERROR,
                      std::string(name) + "[t] must have the shape [batch of step t, " + std::to_string(cols) + "], got " + ShapeStr(arrays[t]));
    }
}

unsigned CellBlocks(int64_t items) {
    int64_t b = (items + 255) / 256;
    const int64_t cap = static_cast<int64_t>(NumCUs()) * 8;
    return static_cast<unsigned>(b > cap ? cap : (b < 1 ? 1 : b));
}

// Layer-directions that advance together are the two directions of a layer or, as a wavefront, all layers of a one-directional network, layer l a step
// behind layer l - 1.  The latter needs the products with the layers' inputs to be part of the steps, which then read twice as much but are fewer: it
// pays to the largest launches tried, four workgroups (32 rows, 8 or 32 units each) to a compute unit (us, forward and backward, products over
// all steps -> in the steps: 2 x 650 LSTM units, 20 rows, 35 steps 1671 -> 1190; 2 x 649, 128 rows 3883 -> 3486; 3 x 600 GRU units, 128 rows 3235 ->
// 2566).  Two directions advance together either way, and only small launches gain (2 x 200 GRU units, 20 rows 806 -> 804; 2 x 400, 64 rows 1971 -> 2118).
bool Narrow(const RnnPlan& pl) {
    const int64_t units = pl.G == 1 ? 32 : 8, rows = (*std::max_element(pl.bt.begin(), pl.bt.end()) + 31) / 32;
    const int64_t jobs = pl.D == 2 ? 2 : pl.L, most = pl.D == 2 ? NumCUs() / 2 : 4 * NumCUs();
    return jobs <= kMaxJobs && rows * ((pl.H + units - 1) / units) * jobs <= most;
}

// Whether a step's products are library calls (on the bfloat16 pipes, in tiles of 128 x 128, where they are large), the x side's over all steps, with a
// launch for the cells: from 1 G multiply-adds of the h side on, for GRU, whose steps work for a fourth gate, from 0.3.  Not for layers that run as a
// wavefront.  us, forward and backward of 6 steps with as many inputs as units, one layer, steps and library calls:
//   GRU  512 rows, 512 units  247 + 400, 177 + 373    LSTM  256 rows, 1024 units  364 + 626, 313 + 604    RNN 1024 rows, 1024 units 418 + 694, 337 + 697
//        256,     1024        384 + 576, 277 + 539          1024,     512        378 + 741, 367 + 682         512,      2048       647 + 1053, 556 + 1027
//        128,     2048        636 + 938, 463 + 931          1024,     1024     1178 + 2010, 850 + 1911
//   and around the lines: GRU 256, 512 133 + 242, 127 + 246; LSTM 384, 768 308 + 691, 294 + 741; RNN 128, 2048 193 + 389, 215 + 367.
bool Wide(const RnnPlan& pl) {
    const double work = static_cast<double>(*std::max_element(pl.bt.begin(), pl.bt.end())) * pl.G * pl.H * pl.H;
    return work >= (pl.mode == kGru ? 3e8 : 1e9) && (pl.L * pl.D == 1 || !Narrow(pl));
}

// f(jobs), for each launch of a pass: the (layer, direction, step) that it runs.  A direction's step s is time step s or T - 1 - s.
struct Turn {
    int layer, direction, s;
};
template <typename F>
void ForEachTurn(const RnnPlan& pl, bool wavefront, int first_layer, int last_layer, F&& f) {
    std::vector<Turn> turns;
    if (wavefront) {
        for (int s = 0; s < pl.T + pl.L - 1; ++s) {
            turns.clear();
            for (int l = std::max(0, s - pl.T + 1); l < pl.L && l <= s; ++l) turns.push_back({l, 0, s - l});
            f(turns);
        }
        return;
    }
    for (int l = first_layer; l <= last_layer; ++l) {
        for (int s = 0; s < pl.T; ++s) {
            turns.clear();
            for (int d = 0; d < pl.D; ++d) turns.push_back({l, d, s});
            f(turns);
        }
    }
}

// ---- forward ----
void RunForward(Pass& pass, const RnnPlan& pl, int activation, const hipcx_array* hx, const hipcx_array* cx, const hipcx_array* const* ws,
                const hipcx_array* const* bs, const hipcx_array* const* xs, const hipcx_array* hy, const hipcx_array* cy,
                const hipcx_array* const* ys, char* reserve) {
    const int64_t B = pl.B, H = pl.H, GH = pl.G * H, DH = pl.D * H, rows = pl.rows;
    const int chains = pl.L * pl.D;
    const bool wide = Wide(pl), narrow = Narrow(pl) && !wide, wavefront = narrow && pl.D == 1;
    std::vector<const float*> wx, wh, bx, bh;  // (the steps read the x side's matrices of narrow networks only, and none of wide ones)
    for (int idx = 0; idx < chains; ++idx) {
        for (int g = 0; g < 2 * pl.G; ++g) {
            const bool read = g < pl.G ? narrow : !wide;
            (g < pl.G ? wx : wh).push_back(read ? Dense(pass, ws[idx * 2 * pl.G + g]) : nullptr);
            (g < pl.G ? bx : bh).push_back(Dense(pass, bs[idx * 2 * pl.G + g]));
        }
    }
    float* const x_all = pass.Take(rows * pl.I);
    std::vector<float*> y_buf;  // outputs of the layers below the top
    for (int l = 0; l + 1 < pl.L; ++l) {
        if (reserve != nullptr) y_buf.push_back(reinterpret_cast<float*>(reserve + pl.r_y[l]));
        else y_buf.push_back(l < 2 || wavefront ? pass.Take(rows * DH) : y_buf[l - 2]);
    }
    float* xw_all[2] = {nullptr, nullptr};
    if (!narrow) {
        for (int d = 0; d < pl.D; ++d) xw_all[d] = pass.Take(rows * GH);
    }
    float* const h0 = pass.Take(chains * B * H);
    std::vector<float*> wx_packed, wh_packed;
    for (int idx = 0; idx < chains && !narrow; ++idx) wx_packed.push_back(PackWeights(pass, pl, ws, idx, 0));
    for (int idx = 0; idx < chains && wide; ++idx) wh_packed.push_back(PackWeights(pass, pl, ws, idx, pl.G));
    float* hw[2] = {nullptr, nullptr};
    for (int d = 0; d < pl.D && wide; ++d) hw[d] = pass.Take(*std::max_element(pl.bt.begin(), pl.bt.end()) * GH);
    // The steps read what earlier ones left in hy, cy and ys, and the caller's inputs where they are.  Results that share memory with each other (one
    // scratch array for every ys[t]) or with an input are kept here until the end.
    float *const y_own = pass.Take(rows * DH), *const h_own = pass.Take(chains * B * H), *const c_own = pl.mode == kLstm ? pass.Take(chains * B * H) : nullptr;
    pass.StartScratch();
    bool own = false, in_order = false;
    if (!pass.dry()) {
        auto same = [](const hipcx_array* a, const hipcx_array* b) { return a->data == b->data && std::equal(a->strides, a->strides + 3, b->strides); };
        std::vector<const hipcx_array*> outs{hy}, ins;
        if (!same(hx, hy)) ins.push_back(hx);  // (a state that is updated in place is copied onto itself)
        outs.insert(outs.end(), ys, ys + pl.T);
        ins.insert(ins.end(), xs, xs + pl.T);
        ins.insert(ins.end(), ws, ws + chains * 2 * pl.G);
        ins.insert(ins.end(), bs, bs + chains * 2 * pl.G);
        if (pl.mode == kLstm) {
            outs.push_back(cy);
            if (!same(cx, cy)) ins.push_back(cx);
        }
        own = AnyShared(outs, ins);
        in_order = own && AnyShared(outs, {});
    }
    auto h_state = [&](int idx) { return own ? Matrix(h_own + idx * B * H, B, H, H) : StateSlice(hy, idx); };
    auto c_state = [&](int idx) { return own ? Matrix(c_own + idx * B * H, B, H, H) : StateSlice(cy, idx); };
    // the steps read rows of xs where they are if their columns are dense; the products over all steps need them in one array
    bool x_in_place = narrow;
    for (int t = 0; t < pl.T; ++t) x_in_place = x_in_place && (xs[t]->strides[1] == 4 || pl.I == 1) && xs[t]->strides[0] % 4 == 0;
    for (int t = 0; t < pl.T && !x_in_place; ++t) pass.Copy(*xs[t], Matrix(x_all + pl.row_start[t] * pl.I, pl.bt[t], pl.I, pl.I));
    for (int idx = 0; idx < chains; ++idx) {
        pass.Copy(StateSlice(hx, idx), Matrix(h0 + idx * B * H, B, H, H));
        pass.Copy(StateSlice(hx, idx), h_state(idx));
        if (pl.mode == kLstm) pass.Copy(StateSlice(cx, idx), c_state(idx));
    }
    pass.FlushCopies();
    // output rows of layer l at step t, direction d's columns, and their stride
    auto y_at = [&](int l, int d, int t, int64_t* stride) {
        if (l + 1 < pl.L || own) {
            *stride = DH;
            return (l + 1 < pl.L ? y_buf[l] : y_own) + pl.row_start[t] * DH + d * H;
        }
        *stride = ys[t]->strides[0] / 4;
        return static_cast<float*>(ys[t]->data) + d * H;
    };
    std::vector<int64_t> seen(chains, 0);  // rows that some step of a layer-direction has held
    auto launch = [&](const std::vector<Turn>& turns) {
        StepArgs a{};
        a.relu = activation == 1;
        a.H = static_cast<int>(H);
        int64_t most = 0;
        for (size_t i = 0; i < turns.size(); ++i) {
            const int l = turns[i].layer, d = turns[i].direction, s = turns[i].s, idx = l * pl.D + d;
            const int t = d == 0 ? s : pl.T - 1 - s;
            const int64_t bt = pl.bt[t], r0 = pl.row_start[t];
            StepJob& j = a.job[i];
            j.bt = static_cast<int>(bt);
            j.in = static_cast<int>(pl.In(l));
            if (narrow && l == 0) {
                j.x = x_in_place ? static_cast<const float*>(xs[t]->data) : x_all + r0 * pl.I;
                j.x_stride = x_in_place ? xs[t]->strides[0] / 4 : pl.I;
            } else if (narrow) {
                j.x = y_at(l - 1, 0, t, &j.x_stride);
            } else {
                j.xw = xw_all[d] + r0 * GH;
            }
            j.h0 = h0 + idx * B * H;
            if (s > 0) {
                const int before = d == 0 ? t - 1 : t + 1;
                j.prev_rows = static_cast<int>(std::min(bt, pl.bt[before]));
                j.h_prev = y_at(l, d, before, &j.h_prev_stride);
                if (const int64_t back = std::min(bt, seen[idx]); back > j.prev_rows) {  // rows that an earlier step held and the last one did not
                    const hipcx_array state = h_state(idx);
                    hipcx_array from = state;
                    from.data = static_cast<char*>(state.data) + j.prev_rows * state.strides[0];
                    from.shape[0] = back - j.prev_rows;
                    pass.Copy(from, Matrix(h0 + (idx * B + j.prev_rows) * H, back - j.prev_rows, H, H));
                }
            }
            seen[idx] = std::max(seen[idx], bt);
            for (int g = 0; g < pl.G; ++g) {
                j.wx[g] = wx[idx * pl.G + g], j.wh[g] = wh[idx * pl.G + g];
                j.bx[g] = bx[idx * pl.G + g], j.bh[g] = bh[idx * pl.G + g];
            }
            j.y = y_at(l, d, t, &j.y_stride);
            const hipcx_array h_out = h_state(idx);
            j.hy = static_cast<float*>(h_out.data), j.hy_row = h_out.strides[0] / 4, j.hy_col = h_out.strides[1] / 4;
            if (pl.mode == kLstm) {
                const hipcx_array c_out = c_state(idx);
                j.cy = static_cast<float*>(c_out.data), j.cy_row = c_out.strides[0] / 4, j.cy_col = c_out.strides[1] / 4;
            }
            if (reserve != nullptr) {
                j.gates = reinterpret_cast<float*>(reserve + pl.r_gates[idx]) + r0 * pl.GR * H;
                j.hprev = reinterpret_cast<float*>(reserve + pl.r_hprev[idx]) + r0 * H;
                j.cprev = pl.mode == kLstm ? reinterpret_cast<float*>(reserve + pl.r_cprev[idx]) + r0 * H : nullptr;
            }
            const int64_t units = pl.G == 1 ? 32 : 8;
            most = std::max(most, (bt + 31) / 32 * ((H + units - 1) / units));
        }
        pass.FlushCopies();
        if (pass.dry()) return;
        VisitMode(pl.mode, [&](auto mode) {
            hipLaunchKernelGGL(RnnStepKernel<decltype(mode)::value>, dim3(static_cast<unsigned>(most), static_cast<unsigned>(turns.size())),
                               dim3(64 * kStepWaves), 0, pass.hip_stream(), a);
        });
        CheckLaunch("rnn_step");
    };
    // the same for wide networks, whose states are in h0 until the end
    auto launch_wide = [&](const std::vector<Turn>& turns) {
        CellArgs a{};
        a.relu = activation == 1;
        a.H = static_cast<int>(H);
        int64_t most = 0;
        for (size_t i = 0; i < turns.size(); ++i) {
            const int l = turns[i].layer, d = turns[i].direction, s = turns[i].s, idx = l * pl.D + d;
            const int t = d == 0 ? s : pl.T - 1 - s;
            const int64_t bt = pl.bt[t], r0 = pl.row_start[t];
            pass.Dot(Matrix(h0 + idx * B * H, bt, H, H), Matrix(wh_packed[idx], H, GH, 1, H), Matrix(hw[d], bt, GH, GH));
            CellJob& j = a.job[i];
            j.bt = static_cast<int>(bt);
            j.xw = xw_all[d] + r0 * GH, j.hw = hw[d];
            for (int g = 0; g < pl.G; ++g) j.bx[g] = bx[idx * pl.G + g], j.bh[g] = bh[idx * pl.G + g];
            j.h = h0 + idx * B * H;
            if (pl.mode == kLstm) {
                const hipcx_array c_out = c_state(idx);
                j.c = static_cast<float*>(c_out.data), j.c_row = c_out.strides[0] / 4, j.c_col = c_out.strides[1] / 4;
            }
            j.y = y_at(l, d, t, &j.y_stride);
            if (reserve != nullptr) {
                j.gates = reinterpret_cast<float*>(reserve + pl.r_gates[idx]) + r0 * pl.GR * H;
                j.hprev = reinterpret_cast<float*>(reserve + pl.r_hprev[idx]) + r0 * H;
                j.cprev = pl.mode == kLstm ? reinterpret_cast<float*>(reserve + pl.r_cprev[idx]) + r0 * H : nullptr;
            }
            most = std::max(most, bt * H);
        }
        if (pass.dry()) return;
        VisitMode(pl.mode, [&](auto mode) {
            hipLaunchKernelGGL(RnnCellKernel<decltype(mode)::value>, dim3(CellBlocks(most), static_cast<unsigned>(turns.size())), dim3(256), 0, pass.hip_stream(), a);
        });
        CheckLaunch("rnn_cell");
    };
    if (narrow) {
        ForEachTurn(pl, wavefront, 0, pl.L - 1, launch);
    } else {
        for (int l = 0; l < pl.L; ++l) {
            const int64_t in = pl.In(l);
            const float* const x_in = l == 0 ? x_all : y_buf[l - 1];
            // the input projection of every step at once
            for (int d = 0; d < pl.D; ++d) {
                pass.Dot(Matrix(x_in, rows, in, in), Matrix(wx_packed[l * pl.D + d], in, GH, 1, in), Matrix(xw_all[d], rows, GH, GH));
            }
            if (wide) ForEachTurn(pl, false, l, l, launch_wide);
            else ForEachTurn(pl, false, l, l, launch);
        }
    }
    if (wide) {
        for (int idx = 0; idx < chains; ++idx) pass.Copy(Matrix(h0 + idx * B * H, B, H, H), h_state(idx));
        pass.FlushCopies();
    }
    if (own) {  // where they share memory one after the other: the last step's outputs and then the states are what is left
        auto hand_out = [&](const hipcx_array& from, const hipcx_array& to) {
            pass.Copy(from, to);
            if (in_order) pass.FlushCopies();
        };
        for (int d = 0; d < pl.D; ++d) {
            for (int s = 0; s < pl.T; ++s) {
                const int t = d == 0 ? s : pl.T - 1 - s;
                hand_out(Matrix(y_own + pl.row_start[t] * DH + d * H, pl.bt[t], H, DH),
                         Matrix(static_cast<float*>(ys[t]->data) + d * H, pl.bt[t], H, ys[t]->strides[0] / 4));
            }
        }
        for (int idx = 0; idx < chains; ++idx) {
            hand_out(h_state(idx), StateSlice(hy, idx));
            if (pl.mode == kLstm) hand_out(c_state(idx), StateSlice(cy, idx));
        }
        pass.FlushCopies();
    }
    pass.CheckFits();
}

// ---- backward ----
// Parts of a gate's units in RnnBackKernel: two workgroups to a compute unit while each has 96 units or more (2 x 650 LSTM units, 20 rows, whole pass:
// one workgroup 1383 us, two 1190, four 1251; from 200 units on, 3 x 200 LSTM units, 128 rows: 2095, from 96 on 1960).
int BackSubs(const RnnPlan& pl, bool wavefront) {
    const int64_t rows = (*std::max_element(pl.bt.begin(), pl.bt.end()) + 31) / 32;
    const int64_t tiles = rows * (wavefront ? 2 * pl.L - 1 : pl.D) * ((pl.H + 31) / 32) * pl.G;
    return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(2 * NumCUs() / tiles, pl.H / 96)));
}

void RunBackward(Pass& pass, const RnnPlan& pl, int activation, const hipcx_array* const* ws, const hipcx_array* const* bs,
                 const hipcx_array* const* xs, const hipcx_array* dhy, const hipcx_array* dcy, const hipcx_array* const* dys, const char* reserve,
                 const hipcx_array* dhx, const hipcx_array* dcx, const hipcx_array* const* dws, const hipcx_array* const* dbs,
                 const hipcx_array* const* dxs) {
    const int64_t B = pl.B, H = pl.H, GH = pl.G * H, DH = pl.D * H, rows = pl.rows;
    const int chains = pl.L * pl.D;
    const bool wide = Wide(pl), wavefront = Narrow(pl) && pl.D == 1 && !wide;
    const int together = wavefront ? pl.L : pl.D;  // layer-directions that advance together
    const int subs = BackSubs(pl, wavefront), splits = wide ? 1 : pl.G * subs;
    const int64_t most_rows = *std::max_element(pl.bt.begin(), pl.bt.end());
    bool shared = false;  // gradients of a layer that overwrite the matrices of one below
    if (!pass.dry()) {
        std::vector<const hipcx_array*> outs(dws, dws + chains * 2 * pl.G);
        shared = AnyShared(outs, std::vector<const hipcx_array*>(ws, ws + chains * 2 * pl.G));
    }
    std::vector<const float*> wx, wh;
    for (int idx = 0; idx < chains; ++idx) {
        for (int g = 0; g < 2 * pl.G; ++g) {
            if (g >= pl.G) wh.push_back(wide ? nullptr : Dense(pass, ws[idx * 2 * pl.G + g], shared));
            else wx.push_back(wavefront && idx > 0 ? Dense(pass, ws[idx * 2 * pl.G + g], shared) : nullptr);
        }
    }
    std::vector<float*> wx_packed(chains, nullptr);  // for the gradients of a layer's input over all steps
    for (int idx = 0; idx < chains; ++idx) {
        if (!wavefront || idx == 0) wx_packed[idx] = PackWeights(pass, pl, ws, idx, 0);
    }
    std::vector<float*> wh_packed;
    for (int idx = 0; idx < chains && wide; ++idx) wh_packed.push_back(PackWeights(pass, pl, ws, idx, pl.G));
    float* x_all = pass.Take(rows * pl.I);
    float* dy_cur = pass.Take(rows * pl.max_in);   // gradient of the current layer's output rows [rows][D*H]
    float* dx_acc = pass.Take(rows * pl.max_in);   // gradient of its input rows [rows][in]
    float* dx_tmp = pl.D == 2 ? pass.Take(rows * pl.max_in) : nullptr;
    std::vector<float*> dgx_all, dgh_all, dh, dc, dh_parts, dx_parts;  // per layer-direction that advances together
    for (int i = 0; i < together; ++i) {
        dgx_all.push_back(pass.Take(rows * GH));
        dgh_all.push_back(pl.mode == kGru ? pass.Take(rows * GH) : dgx_all[i]);
        dh_parts.push_back(pass.Take(splits * most_rows * H));
        dx_parts.push_back(wavefront && i > 0 ? pass.Take(splits * most_rows * H) : nullptr);
    }
    float* const dh_all = pass.Take(chains * B * H);
    float* const dc_all = pl.mode == kLstm ? pass.Take(chains * B * H) : nullptr;
    float* db = pass.Take(chains * 2 * GH);
    pass.StartScratch();
    for (int t = 0; t < pl.T; ++t) pass.Copy(*xs[t], Matrix(x_all + pl.row_start[t] * pl.I, pl.bt[t], pl.I, pl.I));
    for (int t = 0; t < pl.T; ++t) {
        const hipcx_array dst = Matrix(dy_cur + pl.row_start[t] * DH, pl.bt[t], DH, DH);
        if (dys[t] != nullptr) pass.Copy(*dys[t], dst);
        else pass.Zero(dst);
    }
    for (int idx = 0; idx < chains; ++idx) {
        pass.Copy(StateSlice(dhy, idx), Matrix(dh_all + idx * B * H, B, H, H));
        if (pl.mode != kLstm) continue;
        if (dcy != nullptr) pass.Copy(StateSlice(dcy, idx), Matrix(dc_all + idx * B * H, B, H, H));
        else pass.Zero(Matrix(dc_all + idx * B * H, B, H, H));
    }
    pass.FlushCopies();
    std::vector<std::pair<hipcx_array, hipcx_array>> db_copies;
    auto launch_cells = [&](const CellGradArgs& a, size_t jobs) {
        if (pass.dry()) return;
        int64_t cells = 0;
        for (size_t i = 0; i < jobs; ++i) cells = std::max(cells, std::max(a.job[i].bt, a.job[i].part_rows) * H);
        VisitMode(pl.mode, [&](auto mode) {
            hipLaunchKernelGGL(RnnCellGradKernel<decltype(mode)::value>, dim3(CellBlocks(cells), static_cast<unsigned>(jobs)), dim3(256), 0,
                               pass.hip_stream(), a);
        });
        CheckLaunch("rnn_cell_grad");
    };
    // rows that the step behind a layer-direction's next one left parts for (none behind the last)
    std::vector<int> part_rows(together, 0);
    auto slot = [&](const Turn& turn) { return wavefront ? turn.layer : turn.direction; };
    auto cell_state = [&](CellGradJob& j, int idx, int i) {
        j.dh = dh_all + idx * B * H;
        j.dc = pl.mode == kLstm ? dc_all + idx * B * H : nullptr;
        j.parts = dh_parts[i], j.splits = splits, j.part_rows = part_rows[i];
    };
    auto launch = [&](const std::vector<Turn>& turns) {
        CellGradArgs a{};
        BackArgs b{};
        a.relu = activation == 1;
        a.H = b.H = static_cast<int>(H);
        b.G = pl.G, b.subs = subs;
        int64_t most = 0;
        for (size_t n = 0; n < turns.size(); ++n) {
            const int l = turns[n].layer, d = turns[n].direction, i = slot(turns[n]), idx = l * pl.D + d;
            const int s = turns[n].s;
            const int t = d == 0 ? s : pl.T - 1 - s;
            const int64_t bt = pl.bt[t], r0 = pl.row_start[t];
            CellGradJob& j = a.job[n];
            j.bt = static_cast<int>(bt);
            cell_state(j, idx, i);
            if (wavefront && l + 1 < pl.L) {  // the layer above has just left its input's gradient for this step
                j.dy = dx_parts[l + 1], j.dy_stride = H, j.dy_splits = splits, j.dy_part = bt * H;
            } else {
                j.dy = dy_cur + r0 * DH + d * H, j.dy_stride = DH, j.dy_splits = 1;
            }
            j.gates = reinterpret_cast<const float*>(reserve + pl.r_gates[idx]) + r0 * pl.GR * H;
            j.hprev = reinterpret_cast<const float*>(reserve + pl.r_hprev[idx]) + r0 * H;
            j.cprev = pl.mode == kLstm ? reinterpret_cast<const float*>(reserve + pl.r_cprev[idx]) + r0 * H : nullptr;
            j.dgx = dgx_all[i] + r0 * GH;
            j.dgh = dgh_all[i] + r0 * GH;
            // dh of the state before the step: what the cell left there plus dGh . Wh
            BackJob& q = b.job[n];
            q.bt = j.bt;
            q.dgh = j.dgh, q.dgx = j.dgx;
            q.in = wavefront && l > 0 ? static_cast<int>(H) : 0;
            for (int g = 0; g < pl.G; ++g) q.wh[g] = wh[idx * pl.G + g], q.wx[g] = wx[idx * pl.G + g];
            q.dh_parts = dh_parts[i], q.dx_parts = dx_parts[i];
            part_rows[i] = j.bt;
            most = std::max(most, (bt + 31) / 32 * ((H + 31) / 32 + (q.in + 31) / 32) * splits);
        }
        launch_cells(a, turns.size());
        for (size_t n = 0; n < turns.size() && wide; ++n) {
            const BackJob& q = b.job[n];
            pass.Dot(Matrix(q.dgh, q.bt, GH, GH), Matrix(wh_packed[turns[n].layer * pl.D + turns[n].direction], GH, H, H), Matrix(q.dh_parts, q.bt, H, H));
        }
        if (pass.dry() || wide) return;
        hipLaunchKernelGGL(RnnBackKernel, dim3(static_cast<unsigned>(most), static_cast<unsigned>(turns.size())), dim3(64 * kStepWaves), 0,
                           pass.hip_stream(), b);
        CheckLaunch("rnn_back");
    };
    // the forward turns of layers first .. last (all of them as a wavefront), backwards, and what is left of the last parts
    auto run = [&](int first, int last) {
        std::vector<std::vector<Turn>> turns;
        ForEachTurn(pl, wavefront, first, last, [&](const std::vector<Turn>& t) { turns.push_back(t); });
        std::fill(part_rows.begin(), part_rows.end(), 0);
        for (size_t n = turns.size(); n-- > 0;) launch(turns[n]);
        CellGradArgs a{};
        a.H = static_cast<int>(H);
        for (int i = 0; i < together; ++i) cell_state(a.job[i], wavefront ? i : first * pl.D + i, i);
        launch_cells(a, together);
    };
    // parameter gradients of a layer over all rows, and unless `dx` is null those of its input rows there
    auto finish = [&](int l, float* dx) {
        const int64_t in = pl.In(l);
        const float* x_in = l == 0 ? x_all : reinterpret_cast<const float*>(reserve + pl.r_y[l - 1]);
        for (int d = 0; d < pl.D; ++d) {
            const int idx = l * pl.D + d, i = wavefront ? l : d;
            const float* hprev = reinterpret_cast<const float*>(reserve + pl.r_hprev[idx]);
            // dGx[:, g]^T . x and dGh[:, g]^T . h for all gates g in a launch each
            pass.DotEach(Matrix(dgx_all[i], H, rows, 1, GH), H, Matrix(x_in, rows, in, in), dws + idx * 2 * pl.G, pl.G);
            pass.DotEach(Matrix(dgh_all[i], H, rows, 1, GH), H, Matrix(hprev, rows, H, H), dws + idx * 2 * pl.G + pl.G, pl.G);
            // the biases' are column sums of all gates at once; they go to their arrays at the end
            float* const db_x = db + static_cast<int64_t>(idx) * 2 * GH;
            float* const db_h = dgh_all[i] == dgx_all[i] ? db_x : db_x + GH;
            pass.SumRows(Matrix(dgx_all[i], rows, GH, GH), Vector(db_x, GH));
            if (db_h != db_x) pass.SumRows(Matrix(dgh_all[i], rows, GH, GH), Vector(db_h, GH));
            for (int g = 0; g < 2 * pl.G; ++g) {
                db_copies.emplace_back(Vector((g < pl.G ? db_x : db_h) + (g % pl.G) * H, H), *dbs[idx * 2 * pl.G + g]);
            }
            // the second direction adds to the first
            if (dx == nullptr) continue;
            float* const to = d == 0 ? dx : dx_tmp;
            pass.Dot(Matrix(dgx_all[i], rows, GH, GH), Matrix(wx_packed[idx], GH, in, in), Matrix(to, rows, in, in));
            if (d == 1) pass.Add(Matrix(dx, rows, in, in), Matrix(dx_tmp, rows, in, in), Matrix(dx, rows, in, in));
        }
    };
    if (wavefront) {
        run(0, pl.L - 1);
        for (int l = pl.L - 1; l >= 0; --l) finish(l, l == 0 ? dx_acc : nullptr);
        std::swap(dy_cur, dx_acc);
    } else {
        for (int l = pl.L - 1; l >= 0; --l) {
            run(l, l);
            finish(l, dx_acc);
            std::swap(dy_cur, dx_acc);  // the layer below produced these rows
        }
    }
    for (int idx = 0; idx < chains; ++idx) {
        pass.Copy(Matrix(dh_all + idx * B * H, B, H, H), StateSlice(dhx, idx));
        if (pl.mode == kLstm) pass.Copy(Matrix(dc_all + idx * B * H, B, H, H), StateSlice(dcx, idx));
    }
    for (int t = 0; t < pl.T; ++t) pass.Copy(Matrix(dy_cur + pl.row_start[t] * pl.I, pl.bt[t], pl.I, pl.I), *dxs[t]);
    for (const auto& c : db_copies) pass.Copy(c.first, c.second);
    pass.FlushCopies();
    pass.CheckFits();
}

bool FastLstmApplies(const RnnPlan& pl, bool training) { return pl.mode == kLstm && pl.D == 1 && !training && !Narrow(pl); }

}  // namespace
}  // namespace hipcx

using namespace hipcx;

extern "C" {

size_t hipcx_n_step_rnn_reserve_size(int n_layers, int bidirectional, int mode, const hipcx_array* hx, const hipcx_array* const* xs, int n_steps) {
    try {
        return MakePlan(n_layers, bidirectional, mode, hx, xs, n_steps).reserve_total;
    } catch (...) {
        return 0;
    }
}

size_t hipcx_n_step_rnn_workspace_size(int n_layers, int bidirectional, int mode, int training, const hipcx_array* hx, const hipcx_array* const* xs,
                                       int n_steps) {
    try {
        const RnnPlan pl = MakePlan(n_layers, bidirectional, mode, hx, xs, n_steps);
        if (FastLstmApplies(pl, training != 0)) return hipcx_n_step_lstm_workspace_size(n_layers, hx, xs, n_steps);
        // a dry run over stand-ins for the caller's arrays: dense arrays of the right shapes
        std::vector<hipcx_array> w, b, y;
        std::vector<const hipcx_array*> pw, pb, py;
        for (int idx = 0; idx < pl.L * pl.D; ++idx) {
            for (int g = 0; g < 2 * pl.G; ++g) {
                const int64_t cols = g < pl.G ? pl.In(idx / pl.D) : pl.H;
                w.push_back(Matrix(reinterpret_cast<void*>(uintptr_t{1} << 20), pl.H, cols, cols));
                b.push_back(Vector(reinterpret_cast<void*>(uintptr_t{1} << 20), pl.H));
            }
        }
        for (int t = 0; t < pl.T; ++t) y.push_back(Matrix(reinterpret_cast<void*>(uintptr_t{1} << 20), pl.bt[t], pl.D * pl.H, pl.D * pl.H));
        for (auto& a : w) pw.push_back(&a);
        for (auto& a : b) pb.push_back(&a);
        for (auto& a : y) py.push_back(&a);
        char* fake_reserve = training ? reinterpret_cast<char*>(uintptr_t{1} << 30) : nullptr;
        Pass fwd(nullptr, 0, nullptr);
        RunForward(fwd, pl, 0, hx, hx, pw.data(), pb.data(), xs, hx, hx, py.data(), fake_reserve);
        size_t need = fwd.Need();
        if (training) {
            Pass bwd(nullptr, 0, nullptr);
            RunBackward(bwd, pl, 0, pw.data(), pb.data(), xs, hx, hx, py.data(), fake_reserve, hx, hx, pw.data(), pb.data(), xs);
            need = std::max(need, bwd.Need());
        }
        return need + 4096;  // the caller's arrays may be aligned differently from the stand-ins
    } catch (...) {
        return 0;
    }
}

int hipcx_n_step_rnn(int n_layers, int bidirectional, int mode, int activation, const hipcx_array* hx, const hipcx_array* cx,
                     const hipcx_array* const* ws, const hipcx_array* const* bs, const hipcx_array* const* xs, int n_steps, const hipcx_array* hy,
                     const hipcx_array* cy, const hipcx_array* const* ys, void* reserve, size_t reserve_bytes, void* workspace,
                     size_t workspace_bytes, void* stream) {
    return Guard([&] {
        const RnnPlan pl = MakePlan(n_layers, bidirectional, mode, hx, xs, n_steps);
        HIPCX_REQUIRE(activation == 0 || activation == 1, HIPCX_CHAINERX_ERROR, "n_step_rnn: activation must be 0 (tanh) or 1 (relu)");
        CheckParameters(pl, ws, bs, "ws / bs");
        CheckState(pl, hx, "hx");
        CheckState(pl, hy, "hy");
        if (pl.mode == kLstm) {
            CheckState(pl, cx, "cx");
            CheckState(pl, cy, "cy");
        }
        CheckStepArrays(pl, ys, pl.D * pl.H, "ys", false);
        for (int t = 0; t < pl.T; ++t) {
            HIPCX_REQUIRE(ys[t]->strides[1] == 4 && ys[t]->strides[0] % 4 == 0, HIPCX_NOT_IMPLEMENTED_ERROR,
                          "hip n_step_rnn: ys[t] needs unit stride along its last axis");
        }
        HIPCX_REQUIRE(workspace != nullptr && reinterpret_cast<uintptr_t>(workspace) % 256 == 0, HIPCX_CHAINERX_ERROR,
                      "n_step_rnn: workspace must be 256-byte aligned device memory");
        HIPCX_REQUIRE(reserve == nullptr || (reserve_bytes >= pl.reserve_total && reinterpret_cast<uintptr_t>(reserve) % 256 == 0),
                      HIPCX_CHAINERX_ERROR, "n_step_rnn: reserve too small or not 256-byte aligned: need " + std::to_string(pl.reserve_total) + " bytes");
        if (FastLstmApplies(pl, reserve != nullptr)) {
            CheckStatus(hipcx_n_step_lstm(n_layers, hx, cx, ws, bs, xs, n_steps, hy, cy, ys, workspace, workspace_bytes, stream));
            return;
        }
        Pass pass(workspace, workspace_bytes, stream);
        RunForward(pass, pl, activation, hx, cx, ws, bs, xs, hy, cy, ys, static_cast<char*>(reserve));
    });
}

int hipcx_n_step_rnn_backward(int n_layers, int bidirectional, int mode, int activation, const hipcx_array* hx, const hipcx_array* const* ws,
                              const hipcx_array* const* bs, const hipcx_array* const* xs, int n_steps, const hipcx_array* dhy,
                              const hipcx_array* dcy, const hipcx_array* const* dys, const void* reserve, size_t reserve_bytes,
                              const hipcx_array* dhx, const hipcx_array* dcx, const hipcx_array* const* dws, const hipcx_array* const* dbs,
                              const hipcx_array* const* dxs, void* workspace, size_t workspace_bytes, void* stream) {
    return Guard([&] {
        const RnnPlan pl = MakePlan(n_layers, bidirectional, mode, hx, xs, n_steps);
        HIPCX_REQUIRE(activation == 0 || activation == 1, HIPCX_CHAINERX_ERROR, "n_step_rnn: activation must be 0 (tanh) or 1 (relu)");
        CheckParameters(pl, ws, bs, "ws / bs");
        CheckParameters(pl, dws, dbs, "dws / dbs");
        for (int i = 0; i < pl.L * pl.D * 2 * pl.G; ++i) {
            HIPCX_REQUIRE(IsContiguous(dws[i]) && IsContiguous(dbs[i]), HIPCX_NOT_IMPLEMENTED_ERROR, "hip n_step_rnn_backward: dws and dbs must be C-contiguous");
        }
        CheckState(pl, dhy, "dhy");
        CheckState(pl, dhx, "dhx");
        if (pl.mode == kLstm) {
            if (dcy != nullptr) CheckState(pl, dcy, "dcy");
            CheckState(pl, dcx, "dcx");
        }
        CheckStepArrays(pl, dys, pl.D * pl.H, "dys", true);
        CheckStepArrays(pl, dxs, pl.I, "dxs", false);
        HIPCX_REQUIRE(reserve != nullptr && reserve_bytes >= pl.reserve_total, HIPCX_CHAINERX_ERROR,
                      "n_step_rnn_backward: needs the reserve the forward pass filled (" + std::to_string(pl.reserve_total) + " bytes)");
        HIPCX_REQUIRE(workspace != nullptr && reinterpret_cast<uintptr_t>(workspace) % 256 == 0, HIPCX_CHAINERX_ERROR,
                      "n_step_rnn_backward: workspace must be 256-byte aligned device memory");
        Pass pass(workspace, workspace_bytes, stream);
        RunBackward(pass, pl, activation, ws, bs, xs, dhy, dcy, dys, static_cast<const char*>(reserve), dhx, dcx, dws, dbs, dxs);
    });
}

}  // extern "C"
