// Message-passing pressure-correction network: parameters, forward,
// backward, Adam and the training loop.  See gnn.hpp.
#include "gnn.hpp"

#include <algorithm>
#include <cmath>
#include <random>

#include "gnn_kernels.hpp"
#include "la_kernels.hpp"

namespace nodals {

using namespace gnn;
using dev::copy;
using dev::fill;

namespace {
// Blocks of a backward kernel, and so vectors of partial gradients (70 MB):
// 25 to 27 us a layer and 16 us for their sum at 40,320 rows, with 256 blocks
// 31 to 33 and 9; a first call of a new model is as fast with either.
constexpr int kBackBlocks = 512;
constexpr std::size_t kStageByNull = 512 << 10;  // bytes of a host copy from which it goes by the null stream
inline int grid1(long long n) { return (int)((n + 255) / 256); }
}  // namespace

GnnModel::GnnModel(const CellGraph& g, unsigned seed) {
  require(g.n > 0 && (int)g.off.size() == g.n + 1, "GNN graph is empty or malformed");
  n_ = g.n;
  M_ = (n_ + 31) / 32 * 32;
  // backward: at most two blocks a CU, each over its own run of row tiles
  static_assert(kHid == kWidth && kCat == 2 * kWidth && kIn == 16, "the kernels' shapes");
  backGrid_ = dev::xcdGrid(std::min((M_ + kTile - 1) / kTile, kBackBlocks));
  // parameter layout (FP32 master)
  int o = 0;
  oW0_ = o;
  o += kIn * kHid;
  ob0_ = o;
  o += kHid;
  for (int l = 0; l < kLayers; ++l) {
    oW_[l] = o;
    o += kCat * kHid;
    ob_[l] = o;
    o += kHid;
  }
  ow_ = o;
  o += kHid;
  obout_ = o;
  o += 1;
  np_ = o;
  // He-uniform initialisation from a seeded generator; feature rows beyond
  // kFeatures and all biases start at zero.
  std::vector<float> P((std::size_t)np_, 0.0f);
  std::mt19937 rng(seed);
  auto initW = [&](int off, int K, int N, int activeK) {
    const float a = std::sqrt(6.0f / (float)activeK);
    std::uniform_real_distribution<float> U(-a, a);
    for (int k = 0; k < K; ++k)
      for (int n = 0; n < N; ++n) P[(std::size_t)off + (std::size_t)k * N + n] = k < activeK ? U(rng) : 0.0f;
  };
  initW(oW0_, kIn, kHid, kFeatures);
  for (int l = 0; l < kLayers; ++l) {
    initW(oW_[l], kCat, kHid, kCat);
    // residual branches start small so the initial network is close to the
    // encoder-decoder path
    for (int i = 0; i < kCat * kHid; ++i) P[(std::size_t)oW_[l] + i] *= 0.1f;
  }
  initW(ow_, kHid, 1, kHid);
  for (int i = 0; i < kHid; ++i) P[(std::size_t)ow_ + i] *= 0.1f;

  NODALS_HIP(hipSetDevice(0));
  NODALS_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
  off_.upload(g.off);
  std::vector<int> nb(g.nbr);
  if (nb.empty()) nb.push_back(0);
  nbr_.upload(nb);
  P_.upload(P);
  grad_.alloc((std::size_t)np_);
  m_.alloc((std::size_t)np_);
  v_.alloc((std::size_t)np_);
  fill<float>(stream_, np_, m_.data(), 0.0f);
  fill<float>(stream_, np_, v_.data(), 0.0f);
  o16W0_ = 0;
  int o16 = kIn * kHid;
  for (int l = 0; l < kLayers; ++l) {
    o16W_[l] = o16;
    o16 += kCat * kHid;
  }
  w16_.alloc((std::size_t)o16);
  wt16_.alloc((std::size_t)o16);
  const std::size_t M = (std::size_t)M_;
  for (int l = 0; l <= kLayers; ++l) {
    H_[l].alloc(M * kHid);
    mask_[l].alloc(M * 2);
  }
  for (int l = 0; l < kLayers; ++l) Xm_[l].alloc(M * kHid);
  y_.alloc(M);
  d1_.alloc(M * kHid);
  d2a_.alloc(M * kHid);
  d2b_.alloc(M * kHid);
  part_.alloc((std::size_t)backGrid_ * ((std::size_t)np_ + 1));
  lossPart_.alloc((std::size_t)grid1(M_));
  loss_.alloc(1);
  inX_.alloc(M * kIn);  // padding rows stay zero
  inT_.alloc(M);
  fill<float>(stream_, (long long)M_ * kIn, inX_.data(), 0.0f);
  fill<float>(stream_, M_, inT_.data(), 0.0f);
  NODALS_HIP(hipHostMalloc((void**)&hostLoss_, sizeof(float), hipHostMallocCoherent));
  refreshWeights(stream_);
  NODALS_HIP(hipStreamSynchronize(stream_));
}

GnnModel::~GnnModel() {
  if (hostLoss_) (void)hipHostFree(hostLoss_);
  if (stream_) (void)hipStreamDestroy(stream_);
}

void GnnModel::refreshWeights(hipStream_t s) {
  hipLaunchKernelGGL(k_weight_bf16, grid1(np_), 256, 0, s, np_, kLayers, P_.data(), w16_.data(), wt16_.data());
  NODALS_LAUNCHED();
}

// The runtime stages pageable memory through a ring of its own for each
// stream, and the first 16 MB through a new one cost 0.33 ms a MB in page
// faults.  Large copies therefore go by the null stream, whose ring is in use
// since the mesh was uploaded, behind the model's own work; that costs 5 us a
// copy, which small ones do not win back.  First forward and gradient call of
// a new model: 2.0 -> 0.8 ms at 40,320 rows, 6.6 -> 2.1 ms at 115,200; a later
// call 0.62 and 1.3 ms either way.
const float* GnnModel::stage(const float* host, int width, DBuf<float>& d) {
  const std::size_t bytes = sizeof(float) * (std::size_t)n_ * width;
  if (bytes < kStageByNull) {
    NODALS_HIP(hipMemcpyAsync(d.data(), host, bytes, hipMemcpyHostToDevice, stream_));
  } else {
    NODALS_HIP(hipStreamSynchronize(stream_));
    NODALS_HIP(hipMemcpy(d.data(), host, bytes, hipMemcpyHostToDevice));
  }
  return d.data();
}

void GnnModel::getParams(float* host) const {
  NODALS_HIP(hipStreamSynchronize(stream_));
  NODALS_HIP(hipMemcpy(host, P_.data(), sizeof(float) * (std::size_t)np_, hipMemcpyDeviceToHost));
}

void GnnModel::setParams(const float* host) {
  NODALS_HIP(hipStreamSynchronize(stream_));
  NODALS_HIP(hipMemcpy(P_.data(), host, sizeof(float) * (std::size_t)np_, hipMemcpyHostToDevice));
  fill<float>(stream_, np_, m_.data(), 0.0f);
  fill<float>(stream_, np_, v_.data(), 0.0f);
  adamT_ = 0;
  refreshWeights(stream_);
  NODALS_HIP(hipStreamSynchronize(stream_));
}

void GnnModel::forward(hipStream_t s, const float* X, float* y) {
  hipLaunchKernelGGL(k_encode, (M_ / 32 + 3) / 4, 256, 0, s, M_, X, wt16_.data() + o16W0_, P_.data() + ob0_,
                     H_[0].data(), mask_[0].data());
  NODALS_LAUNCHED();
  const int grid = dev::xcdGrid((M_ + kTile - 1) / kTile);
  for (int l = 0; l < kLayers; ++l) {
#define NODALS_LAYER(LAST)                                                                                            \
  hipLaunchKernelGGL((k_layer<LAST>), grid, 256, 0, s, M_, n_, H_[l].data(), off_.data(), nbr_.data(),                \
                     wt16_.data() + o16W_[l], P_.data() + ob_[l], Xm_[l].data(), H_[l + 1].data(),                    \
                     mask_[l + 1].data(), P_.data() + ow_, P_.data() + obout_, X, kSkip, y_.data())
    if (l == kLayers - 1) NODALS_LAYER(true);
    else NODALS_LAYER(false);
#undef NODALS_LAYER
    NODALS_LAUNCHED();
  }
  if (y && y != y_.data()) copy<float>(s, M_, y_.data(), y);
}

void GnnModel::backward(hipStream_t s, const float* X, const float* t, float* loss) {
  float *d2 = d2a_.data(), *d2o = d2b_.data();
#define NODALS_BACK(MODE, L, HP, XM, W, OW, OB)                                                                       \
  hipLaunchKernelGGL((k_layer_back<MODE>), backGrid_, 256, 0, s, M_, n_, y_.data(), t, H_[kLayers].data(),            \
                     P_.data() + ow_, d1_.data(), d2, off_.data(), nbr_.data(), mask_[L].data(), HP, XM, W,           \
                     d1_.data(), d2o, part_.data(), np_, OW, OB, ow_);                                                \
  NODALS_LAUNCHED()
  for (int l = kLayers - 1; l >= 0; --l) {
    if (l == kLayers - 1) {
      NODALS_BACK(kTop, l + 1, H_[l].data(), Xm_[l].data(), w16_.data() + o16W_[l], oW_[l], ob_[l]);
    } else {
      NODALS_BACK(kMiddle, l + 1, H_[l].data(), Xm_[l].data(), w16_.data() + o16W_[l], oW_[l], ob_[l]);
    }
    std::swap(d2, d2o);
  }
  NODALS_BACK(kBottom, 0, X, nullptr, nullptr, oW0_, ob0_);
#undef NODALS_BACK
  hipLaunchKernelGGL(k_grad_sum, (np_ + 1 + 63) / 64, 256, 0, s, backGrid_, np_, part_.data(), grad_.data(), loss);
  NODALS_LAUNCHED();
}

void GnnModel::adamStep(hipStream_t s, float lr) {
  ++adamT_;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.0f - std::pow(b1, (float)adamT_), c2 = 1.0f - std::pow(b2, (float)adamT_);
  hipLaunchKernelGGL(k_adam, grid1(np_), 256, 0, s, np_, kLayers, P_.data(), grad_.data(), m_.data(), v_.data(), lr,
                     b1, b2, eps, c1, c2, w16_.data(), wt16_.data());
  NODALS_LAUNCHED();
}

void GnnModel::reserveSamples(int capacity) {
  require(capacity >= 1, "sample capacity must be >= 1");
  NODALS_HIP(hipStreamSynchronize(stream_));
  if (capacity != cap_) {
    dataX_.alloc((std::size_t)capacity * M_ * kIn);
    dataT_.alloc((std::size_t)capacity * M_);
    fill<float>(stream_, (long long)capacity * M_ * kIn, dataX_.data(), 0.0f);
    fill<float>(stream_, (long long)capacity * M_, dataT_.data(), 0.0f);
    NODALS_HIP(hipStreamSynchronize(stream_));
  }
  cap_ = capacity;
  nSamples_ = 0;
}

int GnnModel::takeSlot() {
  if (nSamples_ >= cap_) return -1;
  return nSamples_++;
}

double GnnModel::train(int epochs, float lr, unsigned seed, std::vector<double>* epochLoss) {
  require(nSamples_ >= 1, "GNN training needs recorded samples");
  require(epochs >= 1, "epochs must be >= 1");
  std::mt19937 rng(seed);
  std::vector<int> order((std::size_t)nSamples_);
  double last = 0.0;
  for (int e = 0; e < epochs; ++e) {
    for (int i = 0; i < nSamples_; ++i) order[(std::size_t)i] = i;
    std::shuffle(order.begin(), order.end(), rng);
    // the per-step squared-error sums accumulate on the device (one slot
    // per step, summed once per epoch)
    if (epochLoss_.size() < (std::size_t)nSamples_) epochLoss_.alloc((std::size_t)nSamples_);
    int q = 0;
    for (int i : order) {
      forward(stream_, sampleX(i), nullptr);
      backward(stream_, sampleX(i), sampleT(i), epochLoss_.data() + q++);
      adamStep(stream_, lr);
    }
    hipLaunchKernelGGL(k_sum, 1, 256, 0, stream_, nSamples_, epochLoss_.data(), loss_.data());
    NODALS_LAUNCHED();
    NODALS_HIP(hipMemcpyAsync(hostLoss_, loss_.data(), sizeof(float), hipMemcpyDeviceToHost, stream_));
    NODALS_HIP(hipStreamSynchronize(stream_));
    last = (double)*hostLoss_ / n_ / nSamples_;
    if (epochLoss) epochLoss->push_back(last);
  }
  return last;
}

double GnnModel::evaluate() {
  require(nSamples_ >= 1, "GNN evaluation needs recorded samples");
  double sum = 0.0;
  for (int i = 0; i < nSamples_; ++i) {
    forward(stream_, sampleX(i), nullptr);
    hipLaunchKernelGGL(k_sq_error, grid1(M_), 256, 0, stream_, n_, y_.data(), sampleT(i), lossPart_.data());
    NODALS_LAUNCHED();
    hipLaunchKernelGGL(k_sum, 1, 256, 0, stream_, grid1(M_), lossPart_.data(), loss_.data());
    NODALS_LAUNCHED();
    NODALS_HIP(hipMemcpyAsync(hostLoss_, loss_.data(), sizeof(float), hipMemcpyDeviceToHost, stream_));
    NODALS_HIP(hipStreamSynchronize(stream_));
    sum += (double)*hostLoss_ / n_;
  }
  return sum / nSamples_;
}

}  // namespace nodals
