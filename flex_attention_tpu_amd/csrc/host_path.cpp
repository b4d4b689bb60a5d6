// The host's path of a prepared call (see _plans.py), forward and backward, as one autograd function in C++: argument blocks from
// a plan, allocations, launches through the C ABI.  What bounds a small call is the host: with the autograd function and both
// calls in Python, a training step of B=1, H=4, S=512, D=64 in float32 took the host 154-163 us (about 50 us of it the autograd
// thread taking up Python, whose caches it finds cold), of which the GPU is busy for 83 us; this way it takes 81 us, what
// the kernels take (bf16, B=1, H=8, S=1024, D=128, causal: 149-162 -> 90 us).
// Python checks the call and finds the plan; nothing here runs under the interpreter's lock.
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>

#include <memory>

#include "flexattn.h"

namespace {

struct Entries {   // of libflexattn.so, which Python has loaded
  decltype(&flexattn_fwd) fwd;
  decltype(&flexattn_fwd_work) fwd_work;
  decltype(&flexattn_fwd_work_bytes) fwd_bytes;
  decltype(&flexattn_bwd) bwd;
  decltype(&flexattn_bwd_dq) bwd_dq;
  decltype(&flexattn_bwd_dkv) bwd_dkv;
  decltype(&flexattn_bwd_delta) bwd_delta;
  decltype(&flexattn_last_error_string) error;
} lib;

void check(int rc) {   // (the exception classes of _lib.check)
  if (rc == FLEXATTN_OK) return;
  const std::string msg = lib.error();
  TORCH_CHECK_VALUE(rc != FLEXATTN_EINVAL, msg);
  TORCH_CHECK_NOT_IMPLEMENTED(rc != FLEXATTN_ENOTSUP, msg);
  TORCH_CHECK(false, "flexattn error ", rc, ": ", msg);
}

// A block map's arrays.  A call that will run a backward keeps them alive until then.
struct Map {
  at::Tensor state, kv_cnt, kv_idx, q_cnt, q_idx;
  int64_t nq, nk, block_q, block_k;
  void put(flexattn_block_map& m) const {
    m.state = static_cast<const uint8_t*>(state.data_ptr());
    m.kv_cnt = static_cast<const int32_t*>(kv_cnt.data_ptr());
    m.kv_idx = static_cast<const int32_t*>(kv_idx.data_ptr());
    m.q_cnt = static_cast<const int32_t*>(q_cnt.data_ptr());
    m.q_idx = static_cast<const int32_t*>(q_idx.data_ptr());
    m.nq = (int32_t)nq;
    m.nk = (int32_t)nk;
    m.block_q = (int32_t)block_q;
    m.block_k = (int32_t)block_k;
  }
};

// Parameter blocks of one combination of shapes, mask and scale; their pointers are written per launch into copies.
struct Plan {
  flexattn_fwd_params fwd;
  flexattn_bwd_params dq, dkv;
};

struct Call : torch::CustomClassHolder {
  std::shared_ptr<const Plan> plan;
  std::shared_ptr<const Map> fwd, dq, dkv;
};

at::Tensor aligned(const at::Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 ? t : t.clone();
}
void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

at::Tensor forward_pass(const Call& call, const at::Tensor& q_, const at::Tensor& k_, const at::Tensor& v_, at::Tensor* l, at::Tensor* m) {
  const c10::OptionalDeviceGuard guard(q_.device());
  const at::Tensor q = aligned(q_), k = aligned(k_), v = aligned(v_);
  at::Tensor o = at::empty(q.sizes(), q.options());
  flexattn_fwd_params p = call.plan->fwd;
  call.fwd->put(p.map);
  p.q = q.data_ptr();
  p.k = k.data_ptr();
  p.v = v.data_ptr();
  p.o = o.data_ptr();
  if (l != nullptr) {
    const auto rows = q.sizes().slice(0, 3);
    *l = at::empty(rows, q.options().dtype(at::kFloat));
    *m = at::empty(rows, q.options().dtype(at::kFloat));
    p.l = l->data_ptr<float>();
    p.m = m->data_ptr<float>();
  }
  const int64_t bytes = lib.fwd_bytes(&p);
  if (bytes > 0) {   // (a small grid: sums of the parts that lists are cut into; freed in the stream's order)
    const at::Tensor work = at::empty({bytes}, q.options().dtype(at::kByte));
    check(lib.fwd_work(&p, work.data_ptr(), bytes, stream_of(q)));
  } else {
    check(lib.fwd(&p, stream_of(q)));
  }
  return o;
}

struct Attention : torch::autograd::Function<Attention> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                            c10::intrusive_ptr<Call> call) {
    at::Tensor l, m;
    at::Tensor o = forward_pass(*call, q, k, v, &l, &m);
    ctx->save_for_backward({q, k, v, o, l, m});
    ctx->saved_data["call"] = c10::IValue::make_capsule(std::move(call));
    return o;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const auto capsule = ctx->saved_data["call"].toCapsule();
    const Call& call = *static_cast<const Call*>(capsule.get());
    const c10::OptionalDeviceGuard guard(saved[0].device());
    const at::Tensor q = aligned(saved[0]), k = aligned(saved[1]), v = aligned(saved[2]), o = aligned(saved[3]);
    const at::Tensor &l = saved[4], &m = saved[5];
    const at::Tensor dout = aligned(grads[0].contiguous());
    TORCH_CHECK_VALUE(dout.sizes() == o.sizes() && dout.scalar_type() == o.scalar_type() && dout.device() == o.device(),
                      "the gradient of the output has another shape, dtype or device than the output");
    const bool want_dq = ctx->needs_input_grad(0), want_dkv = ctx->needs_input_grad(1) || ctx->needs_input_grad(2);
    const at::Tensor delta = at::empty(l.sizes(), l.options());
    at::Tensor dq, dk, dv;
    auto fill = [&](flexattn_bwd_params& p, const Map& map) {
      map.put(p.map);
      p.q = q.data_ptr();
      p.k = k.data_ptr();
      p.v = v.data_ptr();
      p.dout = dout.data_ptr();
      p.l = l.data_ptr<float>();
      p.m = m.data_ptr<float>();
    };
    flexattn_bwd_params pq = call.plan->dq, pkv = call.plan->dkv;
    if (want_dq) {
      dq = at::empty(q.sizes(), q.options());
      fill(pq, *call.dq);
      pq.dq = dq.data_ptr();
      pq.o = o.data_ptr();
      pq.delta_out = delta.data_ptr<float>();
    }
    if (want_dkv) {
      dk = at::empty(k.sizes(), k.options());
      dv = at::empty(v.sizes(), v.options());
      fill(pkv, *call.dkv);
      pkv.delta = delta.data_ptr<float>();
      pkv.dk = dk.data_ptr();
      pkv.dv = dv.data_ptr();
    }
    void* const stream = stream_of(q);
    if (want_dq && want_dkv) {
      check(lib.bwd(&pq, &pkv, stream));
    } else if (want_dq) {
      check(lib.bwd_dq(&pq, stream));
    } else if (want_dkv) {
      check(lib.bwd_delta(o.data_ptr(), dout.data_ptr(), delta.data_ptr<float>(), delta.numel(), pkv.D, pkv.dtype, stream));
      check(lib.bwd_dkv(&pkv, stream));
    }
    return {dq, dk, dv, at::Tensor()};
  }
};

at::Tensor attend(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, std::shared_ptr<const Plan> plan,
                  std::shared_ptr<const Map> fwd, std::shared_ptr<const Map> dq, std::shared_ptr<const Map> dkv) {
  auto call = c10::make_intrusive<Call>();
  call->plan = std::move(plan);
  call->fwd = std::move(fwd);
  call->dq = std::move(dq);
  call->dkv = std::move(dkv);
  if (!(at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad())))
    return forward_pass(*call, q, k, v, nullptr, nullptr);
  return Attention::apply(q, k, v, std::move(call));
}

template <typename T>
T block_of(const py::bytes& b) {
  const std::string s = b;
  TORCH_CHECK(s.size() == sizeof(T), "a parameter block of ", s.size(), " bytes, expected ", sizeof(T));
  T p;
  std::memcpy(&p, s.data(), sizeof(T));
  return p;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, mod) {
  py::class_<Map, std::shared_ptr<Map>>(mod, "Map")
      .def(py::init([](at::Tensor state, at::Tensor kv_cnt, at::Tensor kv_idx, at::Tensor q_cnt, at::Tensor q_idx, int64_t nq, int64_t nk,
                       int64_t block_q, int64_t block_k) {
        return std::make_shared<Map>(Map{state, kv_cnt, kv_idx, q_cnt, q_idx, nq, nk, block_q, block_k});
      }));
  py::class_<Plan, std::shared_ptr<Plan>>(mod, "Plan").def(py::init([](py::bytes fwd, py::bytes dq, py::bytes dkv) {
    return std::make_shared<Plan>(
        Plan{block_of<flexattn_fwd_params>(fwd), block_of<flexattn_bwd_params>(dq), block_of<flexattn_bwd_params>(dkv)});
  }));
  mod.def("attend", &attend, py::call_guard<py::gil_scoped_release>());
  mod.def("bind", [](uintptr_t fwd, uintptr_t fwd_work, uintptr_t fwd_bytes, uintptr_t bwd, uintptr_t bwd_dq, uintptr_t bwd_dkv, uintptr_t bwd_delta, uintptr_t error) {
    lib.fwd = reinterpret_cast<decltype(lib.fwd)>(fwd);
    lib.fwd_work = reinterpret_cast<decltype(lib.fwd_work)>(fwd_work);
    lib.fwd_bytes = reinterpret_cast<decltype(lib.fwd_bytes)>(fwd_bytes);
    lib.bwd = reinterpret_cast<decltype(lib.bwd)>(bwd);
    lib.bwd_dq = reinterpret_cast<decltype(lib.bwd_dq)>(bwd_dq);
    lib.bwd_dkv = reinterpret_cast<decltype(lib.bwd_dkv)>(bwd_dkv);
    lib.bwd_delta = reinterpret_cast<decltype(lib.bwd_delta)>(bwd_delta);
    lib.error = reinterpret_cast<decltype(lib.error)>(error);
  });
}
