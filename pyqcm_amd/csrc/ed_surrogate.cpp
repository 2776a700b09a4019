// ed_surrogate.cpp -- host side of the learned surrogate: parameters, scaling,
// the training loop (Adam on fp32 masters, bf16 copies for the GEMMs) and
// batched inference.  No reference counterpart: pyqcm has no learned model;
// the surrogate proposes VCA / CDMFT candidates that the exact solver verifies.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <numeric>
#include <random>

#include "ed_surrogate.hpp"

namespace ed {

namespace {
// row pitch of the feature-major matrices: whole k-steps of 32
long rows_pitch(int B) { return (B + 31) / 32 * 32; }
int round8(int n) { return (n + 7) / 8 * 8; }

// deterministic standard normals (Box-Muller on a 64-bit Mersenne twister), so
// that an initialization depends on the seed only
struct Normal {
  std::mt19937_64 g;
  bool have = false;
  double keep = 0.0;
  explicit Normal(uint64_t seed) : g(seed) {}
  double u() { return ((g() >> 11) + 0.5) * (1.0 / 9007199254740992.0); }
  double operator()() {
    if (have) {
      have = false;
      return keep;
    }
    const double r = std::sqrt(-2.0 * std::log(u())), th = 6.283185307179586 * u();
    keep = r * std::sin(th);
    have = true;
    return r * std::cos(th);
  }
};

void zero(float *p, size_t n) {
  if (n) ED_HIP(hipMemsetAsync(p, 0, n * sizeof(float), stream()));
}
void zero(bf16_t *p, size_t n) {
  if (n) ED_HIP(hipMemsetAsync(p, 0, n * sizeof(bf16_t), stream()));
}
}  // namespace

Surrogate::Surrogate(int ni, int no, int w, int d, uint64_t seed) : n_in(ni), n_out(no), width(w), depth(d) {
  if (ni < 1 || no < 1 || d < 1 || w < 8 || w % 8) fail(ED_ERR_INVALID, "surrogate: bad layer sizes (width a multiple of 8)");
  Normal nrm(seed);
  layers.resize(d + 1);
  for (int l = 0; l <= d; ++l) {
    Layer &L = layers[l];
    L.in = l == 0 ? ni : w;
    L.out = l == d ? no : w;
    L.in_pad = round8(L.in);
    L.out_pad = round8(L.out);
    L.out32 = (L.out + 31) / 32 * 32;
    const size_t nw = (size_t)L.out_pad * L.in_pad;
    std::vector<float> W(nw, 0.f), b(L.out_pad, 0.f);
    const double sc = 1.0 / std::sqrt((double)L.in);
    for (int o = 0; o < L.out; ++o)
      for (int i = 0; i < L.in; ++i) W[(size_t)o * L.in_pad + i] = (float)(sc * nrm());
    L.W.upload(W);
    L.b.upload(b);
    for (DevBuf<float> *B : {&L.gW, &L.mW, &L.vW}) {
      B->alloc(nw);
      zero(B->p, nw);
    }
    for (DevBuf<float> *B : {&L.gb, &L.mb, &L.vb}) {
      B->alloc(L.out_pad);
      zero(B->p, L.out_pad);
    }
    // (the row-block kernels read up to a layer width past the last row)
    L.Wb.alloc(nw + kMlpSpare);
    zero(L.Wb.p, L.Wb.n);
    L.Wt.alloc((size_t)L.in_pad * L.out32 + kMlpSpare);
    zero(L.Wt.p, L.Wt.n);
  }
  copy_weights();
  // the range of the row-block kernels; other widths, deeper or wider networks
  // run layer by layer
  rows_ok = (w == 64 || w == 128 || w == 256) && d < kMlpLayers && layers[0].in_pad <= w &&
            mlp_rows_lds(w, d, no, true) <= kMlpRowsLds;
  x_mean.assign(ni, 0.0);
  x_std.assign(ni, 1.0);
  y_mean.assign(no, 0.0);
  y_std.assign(no, 1.0);
  loss_w.assign(no, 1.0);
  std::vector<float> lw(layers[d].out_pad, 0.f);
  for (int o = 0; o < no; ++o) lw[o] = 1.f;
  dloss_w.upload(lw);
  sync();
}

size_t Surrogate::n_params() const {
  size_t n = 0;
  for (const Layer &L : layers) n += (size_t)L.out * L.in + L.out;
  return n;
}

void Surrogate::set_scaling(const double *xm, const double *xs, const double *ym, const double *ys, const double *w) {
  for (int i = 0; i < n_in; ++i) {
    if (xs && !(xs[i] > 0.0)) fail(ED_ERR_INVALID, "surrogate: input scales must be positive");
    if (xm) x_mean[i] = xm[i];
    if (xs) x_std[i] = xs[i];
  }
  for (int o = 0; o < n_out; ++o) {
    if (ys && !(ys[o] > 0.0)) fail(ED_ERR_INVALID, "surrogate: output scales must be positive");
    if (w && !(w[o] >= 0.0)) fail(ED_ERR_INVALID, "surrogate: loss weights must be non-negative");
    if (ym) y_mean[o] = ym[o];
    if (ys) y_std[o] = ys[o];
    if (w) loss_w[o] = w[o];
  }
  std::vector<float> lw(layers.back().out_pad, 0.f);
  for (int o = 0; o < n_out; ++o) lw[o] = (float)loss_w[o];
  dloss_w.upload(lw);
  sync();
}

void Surrogate::get_weights(double *w) const {
  size_t k = 0;
  for (const Layer &L : layers) {
    std::vector<float> W = L.W.to_host(), b = L.b.to_host();
    for (int o = 0; o < L.out; ++o)
      for (int i = 0; i < L.in; ++i) w[k++] = W[(size_t)o * L.in_pad + i];
    for (int o = 0; o < L.out; ++o) w[k++] = b[o];
  }
}

void Surrogate::set_weights(const double *w) {
  size_t k = 0;
  for (Layer &L : layers) {
    std::vector<float> W((size_t)L.out_pad * L.in_pad, 0.f), b(L.out_pad, 0.f);
    for (int o = 0; o < L.out; ++o)
      for (int i = 0; i < L.in; ++i) W[(size_t)o * L.in_pad + i] = (float)w[k++];
    for (int o = 0; o < L.out; ++o) b[o] = (float)w[k++];
    L.W.upload(W);
    L.b.upload(b);
    // a new starting point: the optimizer restarts
    zero(L.mW.p, L.mW.n);
    zero(L.vW.p, L.vW.n);
    zero(L.mb.p, L.mb.n);
    zero(L.vb.p, L.vb.n);
  }
  copy_weights();
  adam_t = 0;
  sync();
}

void Surrogate::copy_weights() {
  for (Layer &L : layers) mlp_copies(L.out, L.in, L.in_pad, L.out32, L.W.p, L.Wb.p, L.Wt.p, stream());
}

MlpRows Surrogate::rows_args(int B, const bf16_t *X, const float *T, const int *idx) {
  MlpRows P;
  P.depth = depth;
  P.n_in = n_in;
  P.n_out = n_out;
  P.in_pad = layers[0].in_pad;
  P.out_pad = layers[depth].out_pad;
  P.out32 = layers[depth].out32;
  P.B = B;
  P.Bp = rows_pitch(B);
  for (int l = 0; l <= depth; ++l) {
    P.W[l] = layers[l].Wb.p;
    P.Wt[l] = layers[l].Wt.p;
    P.bias[l] = layers[l].b.p;
  }
  P.X = X;
  P.T = T;
  P.lw = dloss_w.p;
  P.idx = idx;
  P.scale = 2.f / (float)B;
  P.actT = actT.p;
  P.dzT = dzT.p;
  P.db = db.p;
  return P;
}

MlpShape Surrogate::shape() const {
  MlpShape S;
  S.nl = depth + 1;
  for (int l = 0; l <= depth; ++l) {
    const Layer &L = layers[l];
    S.in[l] = L.in;
    S.out[l] = L.out;
    S.aoff[l] = l == 0 ? 0 : n_in + (long)(l - 1) * width;
    S.zoff[l] = (long)l * width;
    S.t0[l + 1] = S.t0[l] + ((L.out + 31) / 32) * ((L.in + 63) / 64);
    S.poff[l + 1] = S.poff[l] + (long)L.out * L.in;
  }
  S.zoff[depth + 1] = (long)depth * width + n_out;
  S.nw = S.poff[depth + 1];
  return S;
}

MlpParams Surrogate::param_table() {
  MlpParams Q = {};
  for (int l = 0; l <= depth; ++l) {
    Layer &L = layers[l];
    Q.W[l] = L.W.p;
    Q.b[l] = L.b.p;
    Q.mW[l] = L.mW.p;
    Q.vW[l] = L.vW.p;
    Q.mb[l] = L.mb.p;
    Q.vb[l] = L.vb.p;
    Q.gW[l] = L.gW.p;
    Q.gb[l] = L.gb.p;
    Q.Wb[l] = L.Wb.p;
    Q.Wt[l] = L.Wt.p;
    Q.in_pad[l] = L.in_pad;
    Q.out32[l] = L.out32;
  }
  return Q;
}

// batch splits of the weight gradients: 512 rows each, at most 4 (12 -> 256 x 4
// -> 641 at a batch of 2 048, gradient + update launch: 1 split 51 + 8 us, 2 28
// + 8, 4 17 + 8, 8 17 + 9, 16 15 + 11)
int Surrogate::rows_splits(int B) const { return std::max(1, std::min(4, B / 512)); }

void Surrogate::ensure_rows(int B) {
  if (B <= cap_rows) return;
  const long Bp = rows_pitch(B), nb = (B + 31) / 32 * 2;
  actT.alloc((size_t)(n_in + depth * width) * Bp);
  dzT.alloc((size_t)(depth * width + n_out) * Bp);
  db.alloc((size_t)(depth * width + n_out) * nb);
  slab.alloc((size_t)rows_splits(B) * shape().nw);
  cap_rows = B;
}

// (loss is the caller's, part of ensure_batch among them: nothing here may move it)
int Surrogate::rows_step(int B, const bf16_t *X, const float *T, const int *idx, float *loss, const MlpAdam *h) {
  ensure_rows(B);
  MlpRows P = rows_args(B, X, T, idx);
  P.loss = loss;
  const MlpShape S = shape();
  const int nb = mlp_rows(P, width, true, stream()), ns = rows_splits(B);
  mlp_wgrad(S, ns, (B + 31) / 32, P.Bp, actT.p, dzT.p, slab.p, stream());
  mlp_update(S, param_table(), h, ns, nb, slab.p, db.p, stream());
  return nb;
}

MlpAdam Surrogate::next_adam() {
  ++adam_t;
  MlpAdam h;
  h.lr = (float)lr;
  h.b1 = (float)beta1;
  h.b2 = (float)beta2;
  h.eps = (float)eps;
  h.c1 = (float)(1.0 - std::pow(beta1, (double)adam_t));
  h.c2 = (float)(1.0 - std::pow(beta2, (double)adam_t));
  return h;
}

void Surrogate::ensure_batch(int B) {
  if (B <= cap_B) return;
  const Layer &L0 = layers[0], &LN = layers.back();
  xb.alloc((size_t)B * L0.in_pad);
  zero(xb.p, xb.n);
  act_b.alloc((size_t)depth * B * width);
  z.alloc((size_t)depth * B * width);
  y.alloc((size_t)B * LN.out_pad);
  t.alloc((size_t)B * LN.out_pad);
  zero(t.p, t.n);
  dz_b.alloc((size_t)B * std::max(width, LN.out_pad));
  zero(dz_b.p, dz_b.n);
  dz2_b.alloc((size_t)B * width);
  part.alloc(1024);
  // split-k partials of the weight gradients: S slabs of the largest layer
  split_S = std::max(1, std::min(8, B / 256));
  size_t wmax = 0, omax = 0;
  for (const Layer &L : layers) {
    wmax = std::max(wmax, (size_t)L.out_pad * L.in_pad);
    omax = std::max(omax, (size_t)L.out_pad);
  }
  split.alloc(std::max((size_t)split_S * wmax, (size_t)mlp_colsum_chunks(B) * omax));
  cap_B = B;
}

// A forward pass alone through the row-block kernel: 4 096 rows a round of 256
// workgroups, each of which reads all weights (about 4 us and 1 us per 17 000
// weights), against a GEMM per layer, about 10 us each at these sizes.  us at
// width, hidden layers, outputs and rows, GEMMs / row blocks: 256 4 641 4 096 45 /
// 26, 8 192 56 / 49, 9 000 66 / 72, 16 384 75 / 97; 256 2 641 4 096 26 / 19, 8 192
// 33 / 35; 256 4 64 12 288 56 / 46, 16 384 61 / 62; 128 8 641 16 384 91 / 80; 128 1
// 641 8 192 18 / 16, 12 288 23 / 23; 64 8 641 16 384 72 / 46.  A training step is
// the faster in row blocks at every size (256 2 641 16 384: 430 / 228).
bool Surrogate::forward_rows(int B) const {
  const long weights = (long)(depth - 1) * width * width + (long)width * n_out;
  const long rounds = (B + 4095) / 4096;
  return use_rows(B) && (rounds == 1 || rounds * (4 + weights / 17000) <= 10L * (depth + 1));
}

void Surrogate::forward(int B, const bf16_t *x) {
  if (forward_rows(B)) {
    MlpRows P = rows_args(B, x, nullptr, nullptr);
    P.y = y.p;
    mlp_rows(P, width, false, stream());
    return;
  }
  for (int l = 0; l <= depth; ++l) {
    const Layer &L = layers[l];
    GemmArgs g;
    g.M = B;
    g.N = L.out;
    g.K = L.in;
    g.A = l == 0 ? x : act_b.p + (size_t)(l - 1) * B * width;
    g.sam = L.in_pad;
    g.sak = 1;
    g.Kpad = L.in_pad;
    g.B = L.Wb.p;
    g.sbk = 1;
    g.sbn = L.in_pad;
    g.bias = L.b.p;
    if (l < depth) {
      g.Cf = z.p + (size_t)l * B * width;
      g.ldc = width;
      g.Cb = act_b.p + (size_t)l * B * width;
      g.ldcb = width;
      mlp_gemm(g, EPI_BIAS_GELU, stream());
    } else {
      g.Cf = y.p;
      g.ldc = L.out_pad;
      mlp_gemm(g, EPI_BIAS, stream());
    }
  }
}

int Surrogate::backward(int B, float *partials) {
  const Layer &LN = layers.back();
  const int nb = mlp_loss_grad(B, n_out, LN.out_pad, y.p, t.p, dloss_w.p, dz_b.p, partials, stream());
  // backward: dZ of the output layer is in dz_b (row pitch out_pad)
  bf16_t *dcur = dz_b.p, *dnext = dz2_b.p;
  int ldcur = LN.out_pad;
  for (int l = depth; l >= 0; --l) {
    Layer &L = layers[l];
    const bf16_t *Aprev = l == 0 ? xb.p : act_b.p + (size_t)(l - 1) * B * width;
    // dW = dZ^T A_prev (split over the batch, fixed-order reduction)
    GemmArgs g;
    g.M = L.out;
    g.N = L.in;
    g.K = B;
    g.Kpad = round8(B);
    g.A = dcur;
    g.sam = 1;
    g.sak = ldcur;
    g.Mpad = ldcur;
    g.B = Aprev;
    g.sbk = L.in_pad;
    g.sbn = 1;
    g.Npad = L.in_pad;
    g.Cf = split.p;
    g.ldc = L.in_pad;
    g.ksplit = split_S;
    g.split_stride = (long)L.out_pad * L.in_pad;
    mlp_gemm(g, EPI_STORE, stream());
    mlp_split_reduce(split_S, L.out, L.in, L.in_pad, g.split_stride, split.p, L.gW.p, stream());
    // the split partials are folded: their buffer holds the column-sum chunks
    mlp_colsum(B, L.out, ldcur, dcur, L.gb.p, split.p, stream());
    if (l == 0) break;
    // dZ_{l-1} = (dZ_l W_l) * gelu'(Z_{l-1})
    GemmArgs h;
    h.M = B;
    h.N = L.in;
    h.K = L.out;
    h.A = dcur;
    h.sam = ldcur;
    h.sak = 1;
    h.Kpad = ldcur;
    h.B = L.Wb.p;
    h.sbk = L.in_pad;
    h.sbn = 1;
    h.Npad = L.in_pad;
    h.Z = z.p + (size_t)(l - 1) * B * width;
    h.ldz = width;
    h.Cb = dnext;
    h.ldcb = width;
    mlp_gemm(h, EPI_GELU_GRAD, stream());
    // the output layer's gradient is no longer needed: the two buffers alternate
    std::swap(dcur, dnext);
    ldcur = width;
  }
  return nb;
}

double Surrogate::loss_and_grad(int B) {
  int nb;
  if (use_rows(B)) {
    nb = rows_step(B, xb.p, t.p, nullptr, part.p, nullptr);
  } else {
    forward(B, xb.p);
    nb = backward(B, part.p);
  }
  std::vector<float> hp(nb);
  part.download(hp.data(), nb);
  return mlp_fold(hp.data(), nb) / B;
}

void Surrogate::adam_step() {
  const MlpAdam h = next_adam();
  for (Layer &L : layers) {
    mlp_adam(L.W.n, L.W.p, L.gW.p, L.mW.p, L.vW.p, L.Wb.p, h.lr, h.b1, h.b2, h.eps, h.c1, h.c2, stream());
    mlp_adam(L.b.n, L.b.p, L.gb.p, L.mb.p, L.vb.p, nullptr, h.lr, h.b1, h.b2, h.eps, h.c1, h.c2, stream());
  }
  if (rows_ok) copy_weights();  // (a batch beyond the row-block kernels: their transposed copies follow)
}

void Surrogate::upload_inputs(int n, const double *x, DevBuf<bf16_t> &dst) const {
  const int ip = layers[0].in_pad;
  std::vector<float> f((size_t)n * ip, 0.f);
  for (int r = 0; r < n; ++r)
    for (int i = 0; i < n_in; ++i) f[(size_t)r * ip + i] = (float)((x[(size_t)r * n_in + i] - x_mean[i]) / x_std[i]);
  DevBuf<float> tmp;
  tmp.upload(f);
  if (dst.n < f.size()) dst.alloc(f.size());
  mlp_to_bf16(f.size(), tmp.p, dst.p, stream());
  sync();
}

void Surrogate::upload_targets(int n, const double *yv, DevBuf<float> &dst) const {
  const int op = layers.back().out_pad;
  std::vector<float> f((size_t)n * op, 0.f);
  for (int r = 0; r < n; ++r)
    for (int o = 0; o < n_out; ++o) f[(size_t)r * op + o] = (float)((yv[(size_t)r * n_out + o] - y_mean[o]) / y_std[o]);
  if (dst.n < f.size()) dst.alloc(f.size());
  dst.upload(f);
  sync();
}

void Surrogate::predict(int n, const double *x, double *yout) {
  const int chunk = 16384, op = layers.back().out_pad;
  for (int r0 = 0; r0 < n; r0 += chunk) {
    const int B = std::min(chunk, n - r0);
    ensure_batch(B);
    upload_inputs(B, x + (size_t)r0 * n_in, xb);
    forward(B, xb.p);
    std::vector<float> h((size_t)B * op);
    y.download(h.data(), h.size());
    for (int r = 0; r < B; ++r)
      for (int o = 0; o < n_out; ++o)
        yout[(size_t)(r0 + r) * n_out + o] = (double)h[(size_t)r * op + o] * y_std[o] + y_mean[o];
  }
}

double Surrogate::loss_grad_host(int n, const double *x, const double *yv, double *grad) {
  if (n < 1) fail(ED_ERR_INVALID, "surrogate: empty batch");
  ensure_batch(n);
  upload_inputs(n, x, xb);
  upload_targets(n, yv, t);
  const double loss = loss_and_grad(n);
  if (grad) {
    size_t k = 0;
    for (const Layer &L : layers) {
      std::vector<float> W = L.gW.to_host(), b = L.gb.to_host();
      for (int o = 0; o < L.out; ++o)
        for (int i = 0; i < L.in; ++i) grad[k++] = W[(size_t)o * L.in_pad + i];
      for (int o = 0; o < L.out; ++o) grad[k++] = b[o];
    }
  }
  return loss;
}

namespace {
// Device time of the steps of sampled epochs (without the shuffles and index
// uploads between epochs), and with it the bound on how far the host queues
// ahead: a sample begins once the last one has run.  One pair of events; a
// record costs 4 us of the stream's time, so not every short epoch has one.
struct EpochClock {
  hipEvent_t e0 = nullptr, e1 = nullptr;
  double ms = 0.0;
  long steps = 0, pending = 0;
  EpochClock() {
    ED_HIP(hipEventCreate(&e0));
    ED_HIP(hipEventCreate(&e1));
  }
  EpochClock(const EpochClock &) = delete;
  ~EpochClock() {
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
  }
  void wait() {
    if (!pending) return;
    ED_HIP(hipEventSynchronize(e1));
    float t = 0.f;
    ED_HIP(hipEventElapsedTime(&t, e0, e1));
    ms += t;
    steps += pending;
    pending = 0;
  }
  void start() { ED_HIP(hipEventRecord(e0, stream())); }
  void stop(long n) {
    ED_HIP(hipEventRecord(e1, stream()));
    pending = n;
  }
};
}  // namespace

std::vector<double> Surrogate::train(int n, const double *x, const double *yv, int epochs, int batch, uint64_t seed,
                                     double *ms_per_step) {
  if (n < 1 || epochs < 0 || batch < 1) fail(ED_ERR_INVALID, "surrogate: bad training arguments");
  batch = std::min(batch, n);
  const int ip = layers[0].in_pad, op = layers.back().out_pad;
  DevBuf<bf16_t> X;
  DevBuf<float> T;
  upload_inputs(n, x, X);
  upload_targets(n, yv, T);
  if (!use_rows(batch)) ensure_batch(batch);
  const int steps = n / batch;  // full batches only: every step sees the same batch size
  std::vector<int> idx(n);
  std::iota(idx.begin(), idx.end(), 0);
  std::mt19937_64 g(seed);
  // the losses of up to 64 epochs (64 MB of partials) stay on the device before the host reads them
  const size_t per_epoch = (size_t)std::max(steps, 1) * 1024;
  const int group = (int)std::max<size_t>(1, std::min<size_t>({64, (size_t)epochs, (size_t(16) << 20) / per_epoch}));
  DevBuf<int> didx(n);
  DevBuf<float> eparts(per_epoch * (size_t)group);
  std::vector<int> nbs((size_t)std::max(steps, 1) * group);
  std::vector<float> hp;
  std::vector<double> hist;
  // a sampled epoch every 32 steps: the host is at most 64 steps (or two epochs)
  // ahead, and sees a cancellation within as many
  const int every = std::max(1, 32 / std::max(steps, 1));
  EpochClock clock;
  for (int ep0 = 0; ep0 < epochs; ep0 += group) {
    const int ne = std::min(group, epochs - ep0);
    for (int ep = 0; ep < ne; ++ep) {
      for (int i = n - 1; i > 0; --i) std::swap(idx[i], idx[(size_t)(g() % (uint64_t)(i + 1))]);
      didx.upload(idx);
      const bool sample = (ep0 + ep) % every == 0;
      if (sample) clock.wait();
      check_cancel();
      if (sample) clock.start();
      for (int s = 0; s < steps; ++s) {
        const int *bi = didx.p + (size_t)s * batch;
        float *lp = eparts.p + per_epoch * (size_t)ep + (size_t)s * 1024;
        int &nb = nbs[(size_t)ep * steps + s];
        if (use_rows(batch)) {
          const MlpAdam h = next_adam();
          nb = rows_step(batch, X.p, T.p, bi, lp, &h);
          continue;
        }
        mlp_gather_bf16(batch, ip, bi, X.p, xb.p, stream());
        mlp_gather_f32(batch, op, bi, T.p, t.p, stream());
        forward(batch, xb.p);
        nb = backward(batch, lp);
        adam_step();
      }
      if (sample) clock.stop(steps);
    }
    hp.resize(per_epoch * (size_t)ne);
    if (steps) eparts.download(hp.data(), per_epoch * (size_t)ne);
    for (int ep = 0; ep < ne; ++ep) {
      double sum = 0.0;
      for (int s = 0; s < steps; ++s)
        sum += mlp_fold(hp.data() + per_epoch * (size_t)ep + (size_t)s * 1024, nbs[(size_t)ep * steps + s]) / batch;
      hist.push_back(steps ? sum / steps : 0.0);
    }
  }
  clock.wait();
  if (ms_per_step) *ms_per_step = clock.steps ? clock.ms / clock.steps : 0.0;
  return hist;
}

void Surrogate::time(int batch, int nrep, double *ms_fwd, double *ms_fb) {
  ensure_batch(batch);
  // inputs: a fixed pattern of normalized values; targets zero
  std::vector<double> x((size_t)batch * n_in);
  for (size_t i = 0; i < x.size(); ++i) x[i] = x_mean[i % n_in] + x_std[i % n_in] * std::sin(0.37 * (double)i);
  upload_inputs(batch, x.data(), xb);
  zero(t.p, (size_t)batch * layers.back().out_pad);
  hipEvent_t e0, e1, e2;
  ED_HIP(hipEventCreate(&e0));
  ED_HIP(hipEventCreate(&e1));
  ED_HIP(hipEventCreate(&e2));
  auto both = [&] {
    if (use_rows(batch)) {
      rows_step(batch, xb.p, t.p, nullptr, part.p, nullptr);
    } else {
      forward(batch, xb.p);
      backward(batch, part.p);
    }
  };
  forward(batch, xb.p);
  both();
  ED_HIP(hipEventRecord(e0, stream()));
  for (int r = 0; r < nrep; ++r) forward(batch, xb.p);
  ED_HIP(hipEventRecord(e1, stream()));
  for (int r = 0; r < nrep; ++r) both();
  ED_HIP(hipEventRecord(e2, stream()));
  ED_HIP(hipEventSynchronize(e2));
  float a = 0.f, b = 0.f;
  ED_HIP(hipEventElapsedTime(&a, e0, e1));
  ED_HIP(hipEventElapsedTime(&b, e1, e2));
  *ms_fwd = a / nrep;
  *ms_fb = b / nrep;
  ED_HIP(hipEventDestroy(e0));
  ED_HIP(hipEventDestroy(e1));
  ED_HIP(hipEventDestroy(e2));
}

}  // namespace ed
