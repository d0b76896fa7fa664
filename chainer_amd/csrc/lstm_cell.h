// The Lstm cell of the routine (CX/routines/connection.cc:396-446).
#pragma once

#include "common.h"

namespace hipcx {

// h and `c_new` from the pre-activations of candidate, input, forget and output gate, in the order of the routine's kernels.  Sigmoid as it composes it
// (CX/routines/activation.cc:74-78): Reciprocal(1 + Exp(-x)) with Reciprocal = 1 / x.  (The float16 chain rounds after every kernel; here the values stay in
// float until they are stored.)
template <typename C>
__device__ __forceinline__ C LstmCell(const C (&g)[4], C c_old, C& c_new) {
    auto exp_of = [](C v) {
        if constexpr (std::is_same_v<C, float>) return expf(v);
        else return exp(v);
    };
    auto tanh_of = [](C v) {
        if constexpr (std::is_same_v<C, float>) return tanhf(v);
        else return tanh(v);
    };
    auto sigmoid = [&](C v) { return C(1) / (C(1) + exp_of(-v)); };
    const C a = tanh_of(g[0]);
    const C i = sigmoid(g[1]);
    const C f = sigmoid(g[2]);
    const C o = sigmoid(g[3]);
    c_new = a * i + f * c_old;
    return o * tanh_of(c_new);
}

}  // namespace hipcx
