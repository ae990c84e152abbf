#include "models/stack_model.h"
#include "absl/strings/str_format.h"
#include "vkl_hip.h"
#include <string.h>

namespace vkllama
{
namespace
{
// tokens of a prompt that go through the layers together; a longer prompt runs in
// portions of this size, which bounds the activation buffers
constexpr int kPortion = 4096;

absl::Status
launched (const char *what, int e)
{
  if (!e)
    return absl::OkStatus ();
  if (e == 1) // hipErrorInvalidValue: rejected before any launch
    return absl::InvalidArgumentError (absl::StrFormat ("%s: shapes rejected by the HIP layer", what));
  return absl::InternalError (absl::StrFormat ("%s: %s", what, vkl_error_string (e)));
}

// a buffer of at least `rows` rows, zeroed when it is made
absl::Status
reserve (Tensor &t, int rows, int width, GPUDevice *dev, DType dtype)
{
  if ((int)t.height () >= rows && (int)t.width () == width && t.dtype () == dtype)
    return absl::OkStatus ();
  t = Tensor (1, rows, width, dev, dtype);
  VKLLAMA_STATUS_OK (t.create ());
  return launched ("clearing a buffer", vkl_memset (t.data (), 0, t.bytes (), dev->stream ()));
}
}

// ---------------------------------------------------------------------------
// layers
// ---------------------------------------------------------------------------
StackBlock::StackBlock (GPUDevice *dev, Command *command, const std::string &name, std::unique_ptr<TokenMixer> mixer,
                        const MixerParams &mp, const FeedForwardParams &ff)
    : dev_ (dev), command_ (command), prefix_ (name), width_ (mp.width), width_p_ (round_up (mp.width, 64)),
      eps_ (mp.eps), dtype_ (mp.dtype), ff_ (ff), mixer_ (std::move (mixer))
{
}

absl::StatusOr<Tensor>
StackBlock::norm_weights_ (const WeightSource &w, const std::string &name)
{
  auto v = w.vector (prefix_ + name, (size_t)width_);
  VKLLAMA_STATUS_OK (v);
  weight_bytes_ += (size_t)width_p_ * 4;
  return upload_vector (dev_, command_, *v, width_p_);
}

absl::Status
StackBlock::norm_product_ (const char *what, Tensor &x, int S, Tensor &norm, Tensor &w, int n,
                           std::vector<vkl_out_seg> const &segs, Buffers &b, int first)
{
  vkl_add_norm_project p = {};
  if (b.back)
    p.x = b.cat.data (), p.xs = (size_t)b.cat_stride, p.w = b.back->data (), p.K = b.back_k;
  b.back = nullptr;
  p.y = (float *)x.data (), p.ys = (size_t)width_p_, p.W = width_;
  p.norm = (const float *)norm.data (), p.eps = eps_, p.h = b.h.data (), p.hs = (size_t)width_p_, p.Wp = width_p_;
  p.w_next = (const uint16_t *)w.data () + (size_t)first * width_p_, p.N = n, p.segs = segs.data (), p.nseg = (int)segs.size ();
  return launched (what, vkl_add_norm_project_bf16w (&p, dtype_ == FP32 ? VKL_TYPE_F32 : VKL_TYPE_BF16, S, dev_->stream ()));
}

absl::Status
StackBlock::keep_ (Tensor &x, int S, size_t offset, int run, Tensor &norm, Tensor &w, Buffers &b)
{
  const TokenMixer::Rows r = mixer_->kept_rows (S, offset);
  auto segs = mixer_->segments (S, offset, run);
  VKLLAMA_STATUS_OK (segs);
  std::vector<vkl_out_seg> kept;
  for (vkl_out_seg s : *segs)
    if (s.n0 >= r.first && s.n0 < r.first + r.n)
      {
        s.n0 -= r.first;
        kept.push_back (s);
      }
  VKLLAMA_STATUS_OK (norm_product_ ("product of what is kept", x, S, norm, w, r.n, kept, b, r.first));
  return mixer_->keep (S, offset, run);
}

absl::Status
StackBlock::finish (Tensor &x, int S, Buffers &b)
{
  if (!b.back)
    return absl::OkStatus ();
  const int type = dtype_ == FP32 ? VKL_TYPE_F32 : VKL_TYPE_BF16;
  float *xp = (float *)x.data ();
  const vkl_out_seg back = { 0, width_, xp, (size_t)width_p_, VKL_TYPE_F32, VKL_ACT_NONE, xp, 0.f };
  const void *w = b.back->data ();
  b.back = nullptr;
  return launched ("layer output product", vkl_project_bf16w (b.cat.data (), type, (size_t)b.cat_stride, w, S, width_,
                                                              b.back_k, &back, 1, dev_->stream ()));
}

ParallelBlock::ParallelBlock (GPUDevice *dev, Command *command, const std::string &name,
                              std::unique_ptr<TokenMixer> mixer, const MixerParams &mp, const FeedForwardParams &ff)
    : StackBlock (dev, command, name, std::move (mixer), mp, ff)
{
  up_row_ = mixer_->in_rows ();
  n_in_ = up_row_ + round_up (ff_.ff, 8);
  ff_col_ = mixer_->out_cols ();
  k_out_ = round_up (ff_col_ + ff_.ff, 64);
}

absl::Status
ParallelBlock::load (const WeightSource &w)
{
  VKLLAMA_STATUS_OK (mixer_->init ());
  VKLLAMA_STATUS_OK (mixer_->load (w, prefix_ + "mix."));
  VKL_TAKE (norm_, norm_weights_ (w, "norm1"));
  PackedMatrix in (n_in_, width_p_), out (width_, k_out_);
  VKLLAMA_STATUS_OK (mixer_->pack_in (w, prefix_ + "mix.", in));
  VKLLAMA_STATUS_OK (mixer_->pack_out (w, prefix_ + "mix.", out));
  if (ff_.ff)
    {
      auto up = w.matrix (prefix_ + "mlp.up", (size_t)ff_.ff, (size_t)width_);
      VKLLAMA_STATUS_OK (up);
      auto down = w.matrix (prefix_ + "mlp.down", (size_t)width_, (size_t)ff_.ff);
      VKLLAMA_STATUS_OK (down);
      in.put (*up, ff_.ff, width_, up_row_);
      out.put (*down, width_, ff_.ff, 0, ff_col_);
    }
  VKL_TAKE (w_in_, in.upload (dev_, command_));
  VKL_TAKE (w_out_, out.upload (dev_, command_));
  weight_bytes_ += w_in_.bytes () + w_out_.bytes ();
  return absl::OkStatus ();
}

absl::Status
ParallelBlock::operator() (Tensor &x, int S, size_t offset, int run, Buffers &b)
{
  const int type = dtype_ == FP32 ? VKL_TYPE_F32 : VKL_TYPE_BF16;
  const size_t esize = dtype_ == FP32 ? 4 : 2, cs = (size_t)b.cat_stride;
  auto segs = mixer_->segments (S, offset, run);
  VKLLAMA_STATUS_OK (segs);
  if (ff_.ff)
    segs->push_back ({ up_row_, ff_.ff, (uint8_t *)b.cat.data () + (size_t)ff_col_ * esize, cs, type, ff_.act, nullptr,
                       0.f });
  VKLLAMA_STATUS_OK (norm_product_ ("layer input product", x, S, norm_, w_in_, n_in_, *segs, b));
  VKLLAMA_STATUS_OK (mixer_->mix (S, offset, run, b.cat.data (), cs));
  b.back = &w_out_, b.back_k = k_out_;
  return absl::OkStatus ();
}

void
ParallelBlock::describe (vkl_stack_layer &l, int run)
{
  mixer_->describe (l, run);
  l.ff = ff_.ff, l.ff_act = ff_.act;
  l.norm = (const float *)norm_.data ();
  l.w_in = w_in_.data (), l.n_in = n_in_, l.up0 = up_row_;
  l.w_out = w_out_.data (), l.k_out = k_out_, l.ff_col = ff_col_;
}

SequentialBlock::SequentialBlock (GPUDevice *dev, Command *command, const std::string &name,
                                  std::unique_ptr<TokenMixer> mixer, const MixerParams &mp,
                                  const FeedForwardParams &ff)
    : StackBlock (dev, command, name, std::move (mixer), mp, ff)
{
  n_in_ = mixer_->in_rows ();
  k_out_ = round_up (mixer_->out_cols (), 64);
  ff_p_ = round_up (ff_.ff, 64);
}

absl::Status
SequentialBlock::load (const WeightSource &w)
{
  VKLLAMA_STATUS_OK (mixer_->init ());
  VKLLAMA_STATUS_OK (mixer_->load (w, prefix_ + "mix."));
  VKL_TAKE (norm1_, norm_weights_ (w, "norm1"));
  PackedMatrix in (n_in_, width_p_), out (width_, k_out_);
  VKLLAMA_STATUS_OK (mixer_->pack_in (w, prefix_ + "mix.", in));
  VKLLAMA_STATUS_OK (mixer_->pack_out (w, prefix_ + "mix.", out));
  VKL_TAKE (w_in_, in.upload (dev_, command_));
  VKL_TAKE (w_out_, out.upload (dev_, command_));
  weight_bytes_ += w_in_.bytes () + w_out_.bytes ();
  if (!ff_.ff)
    return absl::OkStatus ();
  VKL_TAKE (norm2_, norm_weights_ (w, "norm2"));
  auto up = w.matrix (prefix_ + "mlp.up", (size_t)ff_.ff, (size_t)width_);
  VKLLAMA_STATUS_OK (up);
  auto down = w.matrix (prefix_ + "mlp.down", (size_t)width_, (size_t)ff_.ff);
  VKLLAMA_STATUS_OK (down);
  // (up to the padded count: the rows behind put zeros where the product back reads)
  PackedMatrix pu (ff_p_, width_p_), pd (width_, ff_p_);
  pu.put (*up, ff_.ff, width_, 0);
  pd.put (*down, width_, ff_.ff, 0);
  VKL_TAKE (w_up_, pu.upload (dev_, command_));
  VKL_TAKE (w_down_, pd.upload (dev_, command_));
  weight_bytes_ += w_up_.bytes () + w_down_.bytes ();
  return absl::OkStatus ();
}

absl::Status
SequentialBlock::operator() (Tensor &x, int S, size_t offset, int run, Buffers &b)
{
  const int type = dtype_ == FP32 ? VKL_TYPE_F32 : VKL_TYPE_BF16;
  const size_t cs = (size_t)b.cat_stride;
  auto segs = mixer_->segments (S, offset, run);
  VKLLAMA_STATUS_OK (segs);
  VKLLAMA_STATUS_OK (norm_product_ ("mixer input product", x, S, norm1_, w_in_, n_in_, *segs, b));
  VKLLAMA_STATUS_OK (mixer_->mix (S, offset, run, b.cat.data (), cs));
  b.back = &w_out_, b.back_k = k_out_;
  if (!ff_.ff)
    return absl::OkStatus ();
  VKLLAMA_STATUS_OK (norm_product_ ("feed-forward product", x, S, norm2_, w_up_, ff_p_,
                                    { { 0, ff_p_, b.cat.data (), cs, type, ff_.act, nullptr, 0.f } }, b));
  b.back = &w_down_, b.back_k = ff_p_;
  return absl::OkStatus ();
}

void
SequentialBlock::describe (vkl_stack_layer &l, int run)
{
  mixer_->describe (l, run);
  l.ff = ff_.ff, l.ff_act = ff_.act, l.ff_p = ff_p_;
  l.norm = (const float *)norm1_.data ();
  l.w_in = w_in_.data (), l.n_in = n_in_, l.up0 = n_in_;
  l.w_out = w_out_.data (), l.k_out = k_out_, l.ff_col = k_out_;
  if (!ff_.ff)
    return;
  l.norm2 = (const float *)norm2_.data ();
  l.w_up = w_up_.data (), l.w_down = w_down_.data ();
}

// ---------------------------------------------------------------------------
// the model
// ---------------------------------------------------------------------------
StackModel::~StackModel ()
{
  if (gpu_ && gpu_->stream ())
    vkl_stream_sync (gpu_->stream ());
  plan_.reset ();
  blocks_.clear ();
  buf_ = StackBlock::Buffers ();
  embed_ = head_ = embed_norm_ = final_norm_ = x_ = toks_ = rows_ = out_h_ = Tensor ();
  release_buffers_ ();
  command_.reset ();
  delete gpu_;
}

absl::Status
StackModel::init_ (const StackConfig &cfg, int layers, const WeightSource &w, const ModelOptions &options)
{
  cfg_ = cfg;
  ModelOptions opt = options;
  if (opt.max_tokens == 0)
    opt.max_tokens = 4096;
  if (opt.max_tokens > (size_t)1 << 24)
    return absl::InvalidArgumentError ("at most 2^24 cached tokens are supported");
  dtype_ = opt.dtype;
  if (dtype_ != BF16 && dtype_ != FP32)
    return absl::InvalidArgumentError ("this model runs in bf16 or fp32");
  vocab_ = (size_t)cfg_.vocab, maxlen_ = opt.max_tokens;
  width_p_ = round_up (cfg_.width, 64);
  gpu_ = new GPUDevice (opt.device);
  VKLLAMA_STATUS_OK (gpu_->init ());
  command_.reset (new Command (gpu_));
  VKLLAMA_STATUS_OK (command_->init ());

  for (int i = 0; i < (cfg_.tied ? 1 : 2); ++i)
    {
      auto table = w.matrix (i ? "head" : "embed", vocab_, (size_t)cfg_.width);
      VKLLAMA_STATUS_OK (table);
      PackedMatrix pm (cfg_.vocab, width_p_);
      pm.put (*table, cfg_.vocab, cfg_.width, 0);
      VKL_TAKE ((i ? head_ : embed_), pm.upload (gpu_, command_.get ()));
    }
  for (int i = cfg_.embed_norm ? 0 : 1; i < 2; ++i)
    {
      auto v = w.vector (i ? "final.norm" : "embed.norm", (size_t)cfg_.width);
      VKLLAMA_STATUS_OK (v);
      VKL_TAKE ((i ? final_norm_ : embed_norm_), upload_vector (gpu_, command_.get (), *v, width_p_));
    }
  MixerParams common;
  common.width = cfg_.width, common.eps = cfg_.eps, common.maxlen = (int)opt.max_tokens, common.dtype = opt.dtype;
  for (int i = 0; i < layers; ++i)
    {
      common.runs = std::max (1, (int)std::count (cfg_.order.begin (), cfg_.order.end (), i));
      std::unique_ptr<StackBlock> b;
      VKLLAMA_STATUS_OK (make_block_ (i, common, b));
      blocks_.push_back (std::move (b));
      VKLLAMA_STATUS_OK (blocks_.back ()->load (w));
      if (blocks_.back ()->mixer ().state_bytes ())
        stateful_ = true;
      buf_.cat_stride = std::max (buf_.cat_stride, blocks_.back ()->cat_width ());
    }

  vkl_stack_model d = {};
  d.width = cfg_.width, d.width_p = width_p_, d.vocab = cfg_.vocab, d.maxlen = (int)maxlen_;
  d.ctype = dtype_ == FP32 ? VKL_TYPE_F32 : VKL_TYPE_BF16;
  d.eps = cfg_.eps, d.logit_cap = cfg_.logit_softcap, d.embed_scale = cfg_.embed_scale;
  d.embed = embed_.data (), d.head = cfg_.tied ? nullptr : head_.data ();
  d.embed_norm = cfg_.embed_norm ? (const float *)embed_norm_.data () : nullptr;
  d.final_norm = (const float *)final_norm_.data ();
  std::vector<vkl_stack_layer> table;
  std::vector<int> seen (blocks_.size (), 0);
  for (int i : cfg_.order)
    {
      vkl_stack_layer l = {};
      blocks_[(size_t)i]->describe (l, seen[(size_t)i]++);
      table.push_back (l);
    }
  auto plan = std::make_unique<StackPlan> ();
  VKLLAMA_STATUS_OK (plan->build (gpu_, d, table));
  plan_ = std::move (plan);
  return command_->wait ();
}

absl::Status
StackModel::wait_all_ ()
{
  return command_->wait ();
}

// the tokens of a call, where its passes read them: host memory that the GPU sees
absl::Status
StackModel::put_tokens_ (std::vector<uint32_t> const &toks)
{
  // (nothing of a call before may still read there)
  VKLLAMA_STATUS_OK (launched ("waiting for the stream", vkl_stream_sync (gpu_->stream ())));
  if (toks_.width () < toks.size ())
    {
      toks_ = Tensor (1, 1, (int)toks.size (), gpu_, UINT32, true);
      VKLLAMA_STATUS_OK (toks_.create ());
    }
  std::copy (toks.begin (), toks.end (), (uint32_t *)toks_.host ());
  return toks_.flush ();
}

// S tokens from number `first` of the call on through every layer; leaves the residual stream in x_.  last_only: only
// the last token's row of it is wanted.  Behind the layers' last mixing of tokens nothing reads the others, so the last
// layer takes what it keeps of all tokens (a product with a few rows of its matrix) and is the one-token step's layer
// for the last one, whose row it keeps once more.  Passes of four layers, us before / now: 1500 tokens behind 600, Fazinex
// 2048 wide 757 / 627; 2048 tokens, Fuzuvik 4096 wide 2953 / 2528; 300 in 32-bit, 2048 wide 743 / 657.  Recurrences need all
// that feeds them, and stay.
absl::Status
StackModel::pass_ (size_t first, int S, size_t offset, std::vector<float> *streams, bool last_only)
{
  void *s = gpu_->stream ();
  VKLLAMA_STATUS_OK (reserve (x_, S, width_p_, gpu_, FP32));
  VKLLAMA_STATUS_OK (reserve (buf_.h, S, width_p_, gpu_, dtype_));
  VKLLAMA_STATUS_OK (reserve (buf_.cat, S, buf_.cat_stride, gpu_, dtype_));
  const uint32_t *ids = (const uint32_t *)toks_.data () + first;
  float *xp = (float *)x_.data ();
  VKLLAMA_STATUS_OK (launched (
      "embedding", cfg_.embed_norm ? vkl_embed_norm_bf16 (embed_.data (), (uint32_t)vocab_, width_p_, cfg_.width, ids,
                                                          (uint32_t)S, (const float *)embed_norm_.data (), cfg_.eps,
                                                          xp, (size_t)width_p_, s)
                                   : vkl_embed_rows_bf16 (embed_.data (), (uint32_t)vocab_, width_p_, cfg_.width, ids,
                                                          (uint32_t)S, cfg_.embed_scale, xp, (size_t)width_p_, s)));
  std::vector<int> seen (blocks_.size (), 0);
  buf_.back = nullptr; // (of a pass that failed)
  for (size_t n = 0; n < cfg_.order.size (); ++n)
    {
      const size_t i = (size_t)cfg_.order[n];
      if (last_only && n + 1 == cfg_.order.size () && blocks_[i]->can_keep (S, offset))
        {
          VKLLAMA_STATUS_OK (blocks_[i]->keep (x_, S, offset, seen[i], buf_));
          return launched ("last layer", vkl_stack_layer_step (&plan_->desc (), (int)n, xp + (size_t)(S - 1) * width_p_,
                                                               (uint32_t)(offset + (size_t)S - 1), s));
        }
      VKLLAMA_STATUS_OK ((*blocks_[i]) (x_, S, offset, seen[i]++, buf_));
      if (streams || n + 1 == cfg_.order.size ())
        VKLLAMA_STATUS_OK (blocks_[i]->finish (x_, S, buf_));
      if (streams)
        {
          std::vector<float> rows ((size_t)S * width_p_);
          VKLLAMA_STATUS_OK (launched ("download", vkl_memcpy_d2h (rows.data (), x_.data (), rows.size () * 4, s)));
          VKLLAMA_STATUS_OK (launched ("download", vkl_stream_sync (s)));
          for (int r = 0; r < S; ++r)
            streams->insert (streams->end (), rows.begin () + (size_t)r * width_p_,
                             rows.begin () + (size_t)r * width_p_ + cfg_.width);
        }
    }
  return absl::OkStatus ();
}

// logits of those rows of x_ -> out [rows, vocab] (device)
absl::Status
StackModel::logits_ (const std::vector<uint32_t> &rows, float *out)
{
  const int type = dtype_ == FP32 ? VKL_TYPE_F32 : VKL_TYPE_BF16, n = (int)rows.size ();
  void *s = gpu_->stream ();
  if (n == 1 && plan_->usable ())
    return launched ("output product", vkl_stack_logits (&plan_->desc (),
                                                         (const float *)x_.data () + (size_t)rows[0] * width_p_, out, s));
  VKLLAMA_STATUS_OK (reserve (rows_, 1, n, gpu_, UINT32));
  VKLLAMA_STATUS_OK (reserve (out_h_, n, width_p_, gpu_, dtype_));
  VKLLAMA_STATUS_OK (command_->upload (rows.data (), rows.size (), rows_));
  VKLLAMA_STATUS_OK (launched ("final norm",
                               vkl_rmsnorm_f32 ((const float *)x_.data (), (size_t)width_p_,
                                                (const uint32_t *)rows_.data (), n, cfg_.width,
                                                (const float *)final_norm_.data (), cfg_.eps, out_h_.data (), type,
                                                (size_t)width_p_, width_p_, s)));
  const vkl_out_seg seg = { 0, cfg_.vocab, out, vocab_, VKL_TYPE_F32, 0, nullptr, cfg_.logit_softcap };
  return launched ("output product", vkl_project_bf16w (out_h_.data (), type, (size_t)width_p_,
                                                        (cfg_.tied ? embed_ : head_).data (), n, cfg_.vocab, width_p_,
                                                        &seg, 1, s));
}

absl::StatusOr<Tensor>
StackModel::forward_ (std::vector<uint32_t> const &toks, const size_t offset, std::vector<uint32_t> const &rows)
{
  VKLLAMA_STATUS_OK (check_span_ (toks.size (), offset));
  Tensor out (1, (int)std::max<size_t> (rows.size (), 1), (int)vocab_, gpu_, FP32);
  VKLLAMA_STATUS_OK (out.create ());
  VKLLAMA_STATUS_OK (put_tokens_ (toks));
  for (size_t at = 0; at < toks.size (); at += kPortion)
    {
      const int S = (int)std::min<size_t> (kPortion, toks.size () - at);
      // the row of the last token and no other of this portion
      const bool last_only = fused_decode_ && plan_->usable () && S > 1
                             && std::all_of (rows.begin (), rows.end (),
                                             [&] (uint32_t r) { return r < at || r >= at + (size_t)S - 1; })
                             && std::count (rows.begin (), rows.end (), (uint32_t)(at + (size_t)S - 1));
      VKLLAMA_STATUS_OK (pass_ (at, S, offset + at, nullptr, last_only));
      // runs of wanted rows that fall into this portion (in the order asked for)
      for (size_t i = 0; i < rows.size ();)
        {
          std::vector<uint32_t> here;
          const size_t first = i;
          while (i < rows.size () && rows[i] >= at && rows[i] < at + (size_t)S)
            here.push_back (rows[i++] - (uint32_t)at);
          if (here.empty ())
            {
              ++i;
              continue;
            }
          VKLLAMA_STATUS_OK (logits_ (here, (float *)out.data () + first * vocab_));
        }
    }
  return out;
}

absl::StatusOr<std::vector<float> >
StackModel::residual_streams (std::vector<uint32_t> const &toks, size_t offset)
{
  VKLLAMA_STATUS_OK (check_span_ (toks.size (), offset));
  if (toks.size () > (size_t)kPortion)
    return absl::InvalidArgumentError ("residual streams: one portion at most");
  std::vector<float> out;
  VKLLAMA_STATUS_OK (begin_pass_ (offset));
  VKLLAMA_STATUS_OK (put_tokens_ (toks));
  VKLLAMA_STATUS_OK (pass_ (0, (int)toks.size (), offset, &out));
  end_pass_ (offset + toks.size ());
  return out;
}

size_t
StackModel::decode_step_bytes (size_t L) const
{
  size_t n = (cfg_.tied ? embed_ : head_).bytes () + final_norm_.bytes () + (size_t)width_p_ * 2;
  for (int i : cfg_.order)
    {
      TokenMixer &mixer = blocks_[(size_t)i]->mixer ();
      n += blocks_[(size_t)i]->weight_bytes () + mixer.rows_read (L) * mixer.row_bytes () + 2 * mixer.state_bytes ();
    }
  return n;
}
}
