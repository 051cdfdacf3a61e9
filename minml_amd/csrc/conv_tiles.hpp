/*
 * conv_tiles.hpp — products and convolutions of a few thousand rows or fewer: output tiles small enough to occupy the chip, and
 * convolutions whose channel count leaves 128-byte pieces that straddle taps.
 *
 * The 256-row tiles of gemm_dma.hpp give 9 positions of a 128-channel board 8 workgroups; each walks the whole K extent alone, so the
 * launch takes as long as one of 250 positions. Such a launch is bound by that chain (request, wait, multiply, once per piece of K), not
 * by HBM or the matrix cores: what shortens it is more workgroups with less to do per step. Here a workgroup owns 32 x 32, 64 x 64 or
 * 128 x 64 outputs as 16x16 MFMA blocks (bit-identical to the 32x32 blocks of the other
 * engines: a position's result does not depend on the batch it is part of), the operands of the next steps fly directly into a ring of LDS slots, one barrier per slot; the smallest tile takes
 * 256 bytes of K per slot because its two MFMAs per 128 bytes do not cover a barrier (9.1 against 9.8 us at 7200 x 128, K = 1152).
 * The tap of every 16-byte chunk is tracked per lane, so any channel count of whole 16-byte chunks is served, and K past its end reads
 * zeros: gemm_core.hpp's register-staged tiles, which these shapes took before, have one buffer of lookahead.
 *
 * Measured, us per launch, before -> now (tile): int8 3x3, 15x15 positions: 128 channels 9 positions 14.6 -> 5.1 (32 x 32), 32: 14.8 -> 7.1
 * (64 x 64), 96: 15.7 -> 12.1, 128: 16.1 -> 12.1 (128 x 128, gemm_dma.hpp); 256 channels 9: 34.9 -> 7.3, 32: 34.1 -> 13.8, 80: 36.3 -> 25.8;
 * 96 channels 9: 18.8 -> 4.9, 256: 24.4 -> 21.3 (128 x 64), 1024: 79 -> 68; 64 channels 1024: 55 -> 33; 192 channels 1024: 217 -> 162.
 * fp16, 19x19 positions: 5x5 of 256 channels 1: 131 -> 24, 16: 133 -> 52, 64: 141 -> 112; 3x3 of 128 channels 4: 19.7 -> 6.7; 3x3 of 384
 * channels 4: 63 -> 22. fp32 3x3 of 256 channels, 19x19, 1: 541 -> 33, 8: 548 -> 68, 64: 560 -> 260. The order
 * of K is a template parameter: decided at run time it cost the smallest tile 0.6 of 5.7 us.
 */
#ifndef MINML_AMD_CONV_TILES_HPP_
#define MINML_AMD_CONV_TILES_HPP_

#include "common.hpp"
#include "gemm_dma.hpp"

namespace mlhip
{
	/*
	 * 16x16 MFMA blocks. fp16 and int8: one 16-byte fragment per lane and operand (lane l: row l % 16, bytes 16 (l / 16) ... of a k step of
	 * 64 bytes). fp32: k steps of 32 bytes, in which the lanes of quarter q supply elements q / 2 and q / 2 + 2 of the 16-byte half q % 2, so
	 * that the sums run over k in the order 0 4 1 5 2 6 3 7 of the 32x32x2 blocks.
	 */
	template<typename T>
	struct Mfma16Traits;
	template<>
	struct Mfma16Traits<half_t>
	{
			typedef float acc_t;
			typedef float4_t acc_vec;
			typedef uint4_t Fragment;
			static constexpr int STEP = 64;
			__device__ static __forceinline__ int chunk(int quarter)
			{
				return quarter;
			}
			__device__ static __forceinline__ Fragment load(const uint8_t *chunk, int)
			{
				return *reinterpret_cast<const uint4_t*>(chunk);
			}
			__device__ static __forceinline__ void mma(const Fragment &a, const Fragment &b, acc_vec &c)
			{
				c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
			}
	};
	template<>
	struct Mfma16Traits<float>
	{
			typedef float acc_t;
			typedef float4_t acc_vec;
			struct Fragment
			{
					float first, second;
			};
			static constexpr int STEP = 32;
			__device__ static __forceinline__ int chunk(int quarter)
			{
				return quarter & 1;
			}
			__device__ static __forceinline__ Fragment load(const uint8_t *chunk, int quarter)
			{
				const float *src = reinterpret_cast<const float*>(chunk) + (quarter >> 1);
				return Fragment { src[0], src[2] };
			}
			__device__ static __forceinline__ void mma(const Fragment &a, const Fragment &b, acc_vec &c)
			{
				c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.first, b.first, c, 0, 0, 0);
				c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.second, b.second, c, 0, 0, 0);
			}
	};
	template<>
	struct Mfma16Traits<int8_t>
	{
			typedef int acc_t;
			typedef int4_t acc_vec;
			typedef uint4_t Fragment;
			static constexpr int STEP = 64;
			__device__ static __forceinline__ int chunk(int quarter)
			{
				return quarter;
			}
			__device__ static __forceinline__ Fragment load(const uint8_t *chunk, int)
			{
				return *reinterpret_cast<const uint4_t*>(chunk);
			}
			__device__ static __forceinline__ void mma(const Fragment &a, const Fragment &b, acc_vec &c)
			{
				c = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(int4_t, a), __builtin_bit_cast(int4_t, b), c, 0, 0, 0);
			}
	};

	/* the convolution as the product of the im2row matrix [pixels][K] with the weights [N][K]; K = kernel_h * kernel_w * c_bytes bytes */
	struct ConvTileArgs
	{
			const uint8_t *input, *weights;
			int M, N; /* pixels, filters */
			int height, width, kernel_h, kernel_w;
			int c_bytes, k_bytes; /* c_bytes: a multiple of 16 */
			int fill; /* padding byte, 0..255 */
			size_t pixel_bytes; /* between consecutive pixels: c_bytes, or more where several matrices lie side by side */
			int batch = 1; /* matrices: grid's second dimension, with the distances between their operands (bytes) and results (elements) */
			size_t stride_input = 0, stride_weights = 0, stride_out = 0;
	};

	template<int BLOCKS_M_, int BLOCKS_N_, int WAVES_M_, int WAVES_N_, int PIECES_, int SLOTS_>
	struct ConvTileConfig
	{
			static constexpr int BLOCKS_M = BLOCKS_M_, BLOCKS_N = BLOCKS_N_, WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, WAVES = WAVES_M * WAVES_N;
			static constexpr int PIECES = PIECES_; /* 128-byte pieces of a K row per slot, i.e. per barrier */
			static constexpr int SLOTS = SLOTS_, DISTANCE = SLOTS - 1; /* slots requested ahead of the one being consumed */
			static constexpr int BM = 16 * BLOCKS_M * WAVES_M, BN = 16 * BLOCKS_N * WAVES_N;
			static constexpr int A_LOADS = BM / 8 / WAVES, B_LOADS = BN / 8 / WAVES, LOADS = PIECES * (A_LOADS + B_LOADS);
			static constexpr int PIECE_BYTES = (BM + BN) * 128, SLOT_BYTES = PIECES * PIECE_BYTES, LDS_BYTES = SLOTS * SLOT_BYTES;
			static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "8-row blocks must divide evenly over the wavefronts");
			static_assert(WAVES % 2 == 0, "all 8-row blocks of a wavefront share one swizzle, hence one position within the taps");
			static_assert((DISTANCE - 1) * LOADS <= 63 && LDS_BYTES <= 160 * 1024, "queue depth and LDS");
	};

	/* how a launch walks K */
	enum class ConvOrder
	{
		STRADDLING, /* tap by tap, any channel count of whole 16-byte chunks: the tap of every chunk is a lane's own */
		TAPS, /* tap by tap, c_bytes a multiple of 128: a piece of K lies in one tap, which is the same for all lanes */
		SLICES /* the order of gemm_dma_window.hpp: 128 bytes of the channels over all taps, then the next 128; c_bytes a multiple of 128 */
	};
	/* what the kernel divides by, prepared on the host */
	struct ConvTileDivisors
	{
			FastDivisor tiles_n, pixels, width;
			unsigned int tiles;
	};
	/*
	 * A launch over few rows is as long as one wavefront's chain of instructions, so a piece's addresses are few of them: where its tap is the same for all
	 * lanes, a lane keeps the address of its row's first tap, and a load is an addition of the tap's place and
	 * a choice between that address and the padding; nothing is divided by run-time values. Timestamps in the kernel, int8, 9 15x15 positions
	 * of 128 channels, 32 x 32 tiles, per-lane taps / this: until the addresses' parts are there 0.5 us / 0.2, until 12 loads are out 1.2 / 0.6; the network's
	 * launches 4.9 / 4.2 us, of which a launch without work takes 1.65.
	 */
	template<typename T, typename Cfg, ConvOrder ORDER, typename Epilogue>
	__global__ __launch_bounds__(64 * Cfg::WAVES) void kernel_conv_tiles(ConvTileArgs g, ConvTileDivisors by, Epilogue epilogue)
	{
		typedef Mfma16Traits<T> Traits;
		constexpr int DISTANCE = Cfg::DISTANCE;
		constexpr bool UNIFORM = ORDER != ConvOrder::STRADDLING;
		extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
		const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
		const int frag_row = lane & 15, quarter = lane >> 4;
		const unsigned int full = by.tiles & ~7u;
		const unsigned int id = (blockIdx.x < full) ? (blockIdx.x & 7u) * (full >> 3) + (blockIdx.x >> 3) : blockIdx.x;
		uint32_t column_tile;
		const int m_tile = static_cast<int>(fast_divide(id, by.tiles_n, column_tile)) * Cfg::BM, n_tile = static_cast<int>(column_tile) * Cfg::BN;
		const int wave_m = wave / Cfg::WAVES_N, wave_n = wave % Cfg::WAVES_N;
		const size_t matrix = blockIdx.y;
		epilogue.D += matrix * g.stride_out;
		if constexpr (Epilogue::has_c)
		{
			epilogue.C += matrix * g.stride_out;
			if (epilogue.bias != nullptr)
				epilogue.bias += matrix * epilogue.bias_batch_stride;
		}

		/* this lane's rows of the operands, and its place in them: 16 bytes at kb, which lie in tap (i, j) at byte c (for all lanes alike: of the piece) */
		const int chunk = ((lane & 7) ^ dma_swizzle(wave * 8 + (lane >> 3))) * 16;
		const uint8_t *image[Cfg::A_LOADS], *filter[Cfg::B_LOADS]; /* UNIFORM: the address of the chunk in the row's first tap */
		int row_h[Cfg::A_LOADS], row_w[Cfg::A_LOADS];
#pragma unroll
		for (int u = 0; u < Cfg::A_LOADS; u++)
		{
			const int m = min(m_tile + (wave + Cfg::WAVES * u) * 8 + (lane >> 3), g.M - 1);
			uint32_t rest, w;
			const uint32_t b = fast_divide(m, by.pixels, rest);
			row_h[u] = static_cast<int>(fast_divide(rest, by.width, w)) - (g.kernel_h - 1) / 2;
			row_w[u] = static_cast<int>(w) - (g.kernel_w - 1) / 2;
			image[u] = g.input + matrix * g.stride_input + static_cast<size_t>(b) * by.pixels.divisor * g.pixel_bytes;
			if constexpr (UNIFORM)
				image[u] += static_cast<ptrdiff_t>(row_h[u] * g.width + row_w[u]) * static_cast<ptrdiff_t>(g.pixel_bytes) + chunk;
		}
#pragma unroll
		for (int u = 0; u < Cfg::B_LOADS; u++)
			filter[u] = g.weights + matrix * g.stride_weights + static_cast<size_t>(min(n_tile + (wave + Cfg::WAVES * u) * 8 + (lane >> 3), g.N - 1)) * g.k_bytes + (UNIFORM ? chunk : 0);
		int kb = UNIFORM ? 0 : chunk;
		int tap_i = 0, tap_j = 0, c = kb;
		const auto settle = [&]()
		{
			while (c >= g.c_bytes)
			{
				c -= g.c_bytes;
				if (++tap_j == g.kernel_w)
				{
					tap_j = 0;
					tap_i++;
				}
			}
		};
		if constexpr (!UNIFORM)
			settle();
		/* UNIFORM: bytes from the first tap to the piece's */
		ptrdiff_t place = 0;
		const ptrdiff_t pixel = static_cast<ptrdiff_t>(g.pixel_bytes), next_row = static_cast<ptrdiff_t>(g.width - g.kernel_w) * pixel;
		const auto next_piece = [&]()
		{
			if constexpr (ORDER == ConvOrder::SLICES)
			{
				kb += g.c_bytes;
				place += pixel;
				if (++tap_j == g.kernel_w)
				{
					tap_j = 0;
					place += next_row;
					if (++tap_i == g.kernel_h)
					{
						tap_i = 0;
						kb += 128 - g.k_bytes;
						c += 128;
						place = c;
					}
				}
			}
			else if constexpr (ORDER == ConvOrder::TAPS)
			{
				kb += 128;
				c += 128;
				place += 128;
				if (c == g.c_bytes)
				{
					c = 0;
					place += pixel - g.c_bytes;
					if (++tap_j == g.kernel_w)
					{
						tap_j = 0;
						tap_i++;
						place += next_row;
					}
				}
			}
			else
			{
				kb += 128;
				c += 128;
				settle();
			}
		};
		const int steps = (g.k_bytes + Cfg::PIECES * 128 - 1) / (Cfg::PIECES * 128);
		const uint8_t *const fill = &dma_pad_table.bytes[g.fill][0], *const zeros = &dma_pad_table.bytes[0][0];
		const auto request = [&](int step)
		{
			uint8_t *slot = lds + (step % Cfg::SLOTS) * Cfg::SLOT_BYTES;
#pragma unroll
			for (int p = 0; p < Cfg::PIECES; p++)
			{
				uint8_t *const a_slot = slot + p * Cfg::PIECE_BYTES + wave * 1024, *const b_slot = a_slot + Cfg::BM * 128;
				const auto load = [](const uint8_t *src, uint8_t *dst) __attribute__((always_inline))
				{
					__builtin_amdgcn_global_load_lds((global_ptr_t) src, (lds_ptr_t) dst, 16, 0, 0);
				};
				const bool in_k = (ORDER == ConvOrder::SLICES) ? c < g.c_bytes : kb < g.k_bytes;
				if (!UNIFORM || in_k)
				{
#pragma unroll
					for (int u = 0; u < Cfg::A_LOADS; u++)
					{
						const int x = row_h[u] + tap_i, y = row_w[u] + tap_j;
						const bool inside = static_cast<unsigned int>(x) < static_cast<unsigned int>(g.height)
								&& static_cast<unsigned int>(y) < static_cast<unsigned int>(g.width);
						if constexpr (UNIFORM)
							load(inside ? image[u] + place : fill, a_slot + Cfg::WAVES * u * 1024);
						else
							load(!in_k ? zeros : inside ? image[u] + static_cast<size_t>(x * g.width + y) * g.pixel_bytes + c : fill, a_slot + Cfg::WAVES * u * 1024);
					}
#pragma unroll
					for (int u = 0; u < Cfg::B_LOADS; u++)
						load((UNIFORM || in_k) ? filter[u] + kb : zeros, b_slot + Cfg::WAVES * u * 1024);
				}
				else
				{ /* past the end of K both operands read zeros */
#pragma unroll
					for (int u = 0; u < Cfg::A_LOADS; u++)
						load(zeros, a_slot + Cfg::WAVES * u * 1024);
#pragma unroll
					for (int u = 0; u < Cfg::B_LOADS; u++)
						load(zeros, b_slot + Cfg::WAVES * u * 1024);
				}
				next_piece();
			}
		};
		static_for<DISTANCE>([&](auto s)
		{
			if (decltype(s)::value < steps)
				request(decltype(s)::value);
		});

		int a_first[Cfg::BLOCKS_M], b_first[Cfg::BLOCKS_N]; /* this lane's fragment of a piece's first k step, of the others by XOR */
#pragma unroll
		for (int i = 0; i < Cfg::BLOCKS_M; i++)
		{
			const int row = wave_m * 16 * Cfg::BLOCKS_M + 16 * i + frag_row;
			a_first[i] = row * 128 + ((Traits::chunk(quarter) ^ dma_swizzle(row)) * 16);
		}
#pragma unroll
		for (int j = 0; j < Cfg::BLOCKS_N; j++)
		{
			const int row = wave_n * 16 * Cfg::BLOCKS_N + 16 * j + frag_row;
			b_first[j] = (Cfg::BM + row) * 128 + ((Traits::chunk(quarter) ^ dma_swizzle(row)) * 16);
		}
		typename Traits::acc_vec acc[Cfg::BLOCKS_M][Cfg::BLOCKS_N];
#pragma unroll
		for (int i = 0; i < Cfg::BLOCKS_M; i++)
#pragma unroll
			for (int j = 0; j < Cfg::BLOCKS_N; j++)
				acc[i][j] = typename Traits::acc_vec { 0, 0, 0, 0 };
		const auto multiply = [&](int step)
		{
			const uint8_t *slot = lds + (step % Cfg::SLOTS) * Cfg::SLOT_BYTES;
			constexpr int PER_PIECE = 128 / Traits::STEP, K_STEPS = Cfg::PIECES * PER_PIECE;
			typename Traits::Fragment a[K_STEPS][Cfg::BLOCKS_M], b[K_STEPS][Cfg::BLOCKS_N];
#pragma unroll
			for (int t = 0; t < K_STEPS; t++)
			{
				const uint8_t *piece = slot + (t / PER_PIECE) * Cfg::PIECE_BYTES;
#pragma unroll
				for (int i = 0; i < Cfg::BLOCKS_M; i++)
					a[t][i] = Traits::load(piece + (a_first[i] ^ ((t % PER_PIECE) * Traits::STEP)), quarter);
#pragma unroll
				for (int j = 0; j < Cfg::BLOCKS_N; j++)
					b[t][j] = Traits::load(piece + (b_first[j] ^ ((t % PER_PIECE) * Traits::STEP)), quarter);
			}
#pragma unroll
			for (int t = 0; t < K_STEPS; t++)
#pragma unroll
				for (int i = 0; i < Cfg::BLOCKS_M; i++)
#pragma unroll
					for (int j = 0; j < Cfg::BLOCKS_N; j++)
						Traits::mma(b[t][j], a[t][i], acc[i][j]);
		};
		/* step s is readable once its loads have landed in every wavefront; the same barrier frees the slot of step s - 1 */
		int s = 0;
		for (; s + DISTANCE < steps; s++)
		{
			wait_lgkmcnt<0>();
			wait_vmcnt<(DISTANCE - 1) * Cfg::LOADS>();
			barrier_no_fence();
			request(s + DISTANCE);
			multiply(s);
		}

		/* lane l, register r of block (i, j): m = 16 i + l % 16, n = 16 j + 4 (l / 16) + r; the side inputs fly under the last steps */
		const int m0 = m_tile + wave_m * 16 * Cfg::BLOCKS_M + frag_row, n0 = n_tile + wave_n * 16 * Cfg::BLOCKS_N + 4 * quarter;
		typename Epilogue::Column column[Cfg::BLOCKS_N];
		typename Epilogue::Extra extra[Cfg::BLOCKS_M][Cfg::BLOCKS_N];
		/* the last DISTANCE steps (or all of them, if fewer): nothing more is requested */
		static_for<DISTANCE>([&](auto index)
		{
			constexpr int left = DISTANCE - 1 - decltype(index)::value; /* steps still in flight behind this one */
			if (left < steps)
			{
				wait_vmcnt<left * Cfg::LOADS>();
				barrier_no_fence();
				if constexpr (left == 0)
					if (epilogue.vectorized)
					{
#pragma unroll
						for (int j = 0; j < Cfg::BLOCKS_N; j++)
						{
							const int n = n0 + 16 * j;
							column[j] = epilogue.load_column(n < g.N ? n : 0);
							if (epilogue.has_extra())
#pragma unroll
								for (int i = 0; i < Cfg::BLOCKS_M; i++)
									extra[i][j] = epilogue.load_extra(min(m0 + 16 * i, g.M - 1), n < g.N ? n : 0);
						}
					}
				multiply(steps - 1 - left);
			}
		});
#pragma unroll
		for (int i = 0; i < Cfg::BLOCKS_M; i++)
#pragma unroll
			for (int j = 0; j < Cfg::BLOCKS_N; j++)
			{
				const int m = m0 + 16 * i, n = n0 + 16 * j;
				if (m >= g.M || n >= g.N)
					continue;
				const typename Traits::acc_t vals[4] = { acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3] };
				if (epilogue.vectorized)
					epilogue.apply(m, n, vals, column[j], extra[i][j]);
				else
					epilogue(m, n, vals);
			}
	}

	template<typename T, typename Cfg, ConvOrder ORDER, typename Epilogue>
	inline void launch_conv_tiles_as(hipStream_t stream, const ConvTileArgs &g, const Epilogue &epilogue)
	{
		auto kernel = kernel_conv_tiles<T, Cfg, ORDER, Epilogue>;
		ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), Cfg::LDS_BYTES);
		const int tiles_m = ceil_div(g.M, Cfg::BM), tiles_n = ceil_div(g.N, Cfg::BN);
		const ConvTileDivisors by { make_fast_divisor(tiles_n), make_fast_divisor(static_cast<uint32_t>(g.height) * g.width), make_fast_divisor(g.width),
				static_cast<unsigned int>(tiles_m) * tiles_n };
		hipLaunchKernelGGL(kernel, dim3(by.tiles, g.batch), dim3(64 * Cfg::WAVES), Cfg::LDS_BYTES, stream, g, by, epilogue);
	}

	typedef ConvTileConfig<1, 1, 2, 2, 2, 4> ConvTile32; /* 64 KB of LDS: two workgroups per compute unit */
	typedef ConvTileConfig<1, 2, 4, 2, 1, 3> ConvTile64; /* 48 KB: three */
	typedef ConvTileConfig<2, 2, 4, 2, 1, 2> ConvTile128x64; /* 48 KB: three */
	typedef DmaTileConfig<128, 128, 2, 2, 2, 2, 2> DmaTile128; /* 64 KB: two */

	inline ConvTileArgs dense_tile_args(const DenseDmaRows &a, const DenseDmaRows &b, int M, int N, int k_bytes)
	{
		const size_t row_bytes = (a.row_stride_bytes != 0) ? a.row_stride_bytes : k_bytes;
		return ConvTileArgs { a.base, b.base, M, N, 1, M, 1, 1, k_bytes, k_bytes, 0, row_bytes };
	}
	inline ConvTileArgs conv_tile_args(const void *input, const void *weights, int M, int N, int height, int width, int kernel_h, int kernel_w, size_t c_bytes, int fill)
	{
		return ConvTileArgs { reinterpret_cast<const uint8_t*>(input), reinterpret_cast<const uint8_t*>(weights), M, N, height, width, kernel_h, kernel_w,
				static_cast<int>(c_bytes), static_cast<int>(c_bytes * kernel_h * kernel_w), fill, c_bytes };
	}
	inline long long tiles_of(const ConvTileArgs &g, int rows, int columns)
	{
		return static_cast<long long>(ceil_div(g.M, rows)) * ceil_div(g.N, columns) * g.batch;
	}
	/*
	 * The two smallest shapes, while all their workgroups are resident at once (a second round costs more than the larger tile's longer
	 * chain: 552 tiles of 32 x 32 for 1444 x 384 at K = 6912 take 27.6 us, 138 of 64 x 64 take 21.8; 512 of them for 2025 x 256 take 7.3
	 * against 9.8; 900 tiles of 64 x 64 for 14400 x 256 at K = 2304 take 25 against 18 us of 128 x 128 tiles, 724 of them level).
	 */
	template<typename T, ConvOrder ORDER = ConvOrder::TAPS, typename Epilogue>
	inline bool try_launch_small_tiles(hipStream_t stream, const ConvTileArgs &g, const Epilogue &epilogue)
	{
		const int units = device_compute_units();
		if (tiles_of(g, 32, 32) <= 2LL * units)
			launch_conv_tiles_as<T, ConvTile32, ORDER>(stream, g, epilogue);
		else if (tiles_of(g, 64, 64) <= 3LL * units)
			launch_conv_tiles_as<T, ConvTile64, ORDER>(stream, g, epilogue);
		else
			return false;
		return true;
	}
	/*
	 * Products whose K pieces of 128 bytes each lie within one tap (a_loader, b_loader and g name the same operands): the shapes between
	 * the smallest ones and the 256-row tiles.
	 *   fp16, int8: 128 x 128 tiles of gemm_dma.hpp, resident two per compute unit, while there is no second round of them (256 channels
	 *     at K = 2304, 450 tiles: 28.4 against 38.0 us, 900 tiles: 53.5 against 43.6); at most 128 columns, where the tile is only half of
	 *     the 256-row one, up to one per compute unit (225 tiles 12.1 against 16.1 us, 450 tiles 18.8 against 18.0)
	 *   fp32: the matrix pipe is the limit and an idle compute unit costs most: 128 x 64 tiles while the 256-row tiles leave a quarter of
	 *     the units idle (46208 x 128, 181 tiles of 256 x 128: 139 against 157 us; 23104 x 256, 91 tiles of 256 x 256: 260 against 560)
	 */
	template<typename T, typename ALoader, typename Epilogue>
	inline bool try_launch_fewer_rows(hipStream_t stream, const ALoader &a_loader, const DenseDmaRows &b_loader, const ConvTileArgs &g, const Epilogue &epilogue)
	{
		if (g.batch > 65535 || g.k_bytes == 0) /* without taps no step of K would fetch the side inputs; the other engine's tail does */
			return false;
		if (try_launch_small_tiles<T>(stream, g, epilogue))
			return true;
		const int units = device_compute_units();
		if (sizeof(T) == 4)
		{
			if (tiles_of(g, 256, g.N > 128 ? 256 : g.N > 64 ? 128 : 64) * 4 > units * 3LL)
				return false;
			launch_conv_tiles_as<T, ConvTile128x64, ConvOrder::TAPS>(stream, g, epilogue);
			return true;
		}
		if constexpr (sizeof(T) < 4)
		{
			if (g.N <= 64 || tiles_of(g, 128, 128) > (g.N > 128 ? 2LL : 1LL) * units)
				return false;
			launch_gemm_dma_as<T, DmaTile128>(stream, a_loader, b_loader, g.M, g.N, g.k_bytes, g.batch, g.stride_input, g.stride_weights, g.stride_out, epilogue);
		}
		return true;
	}
	/*
	 * Convolutions whose 128-byte pieces straddle taps. The register-staged 128 x 128 tiles (gemm_core.hpp) remain for pixels of 16 bytes of int8, more than 64
	 * columns and more than 8 tiles per unit, where storing is most of the work and the wider tile gathers every pixel, which one 16-byte load per tap is, once per
	 * 128 columns; and beyond 2^32 threads of these tiles, the most that a launch can have: theirs are a quarter as many. us, these / register-staged:
	 *   int8 3x3 without residual, 16 -> 128 channels: 115200 pixels (1800 tiles) 20.2 / 20.5, 159975 (2500) 24.2 / 23.0; 16 -> 256: 79875 (2500) 24.4 / 23.0, 230400 (7200)
	 *   60.5 / 55.3 (with residual 75.7 / 68.7, from memory 83.2 / 90.3); 5x5 16 -> 256: 230400 82.2 / 75.7; but 16 -> 64: 230400 20.2 / 27.9; 32 -> 256: 39825 14.6 / 16.8, 79875 25.4 /
	 *   27.0, 230400 63.8 / 65.6 (with residual from memory 90.1 / 101.0); 48 -> 256: 230400 72.4 / 76.3
	 *   fp16 3x3, 8 -> 64: 230400 20.2 / 33.9; 8 -> 256: 39825 15.2 / 18.1, 460800 111 / 133; 24 -> 256: 230400 70.7 / 90.4; fp32 4 -> 256: 39825 24.2 / 25.4, 460800 208 / 227;
	 *   12 -> 128: 230400 89 / 98; with residual 1.2 to 2.1 times as long throughout
	 */
	inline bool stays_register_staged(const ConvTileArgs &g, int element_size)
	{
		const long long tiles = tiles_of(g, 128, 64);
		return (element_size == 1 && g.c_bytes <= 16 && g.k_bytes <= 512 && g.N > 64 && tiles > 8LL * device_compute_units())
				|| tiles * 64 * ConvTile128x64::WAVES > 0xffffffffLL;
	}
	template<typename T, typename Epilogue>
	inline bool try_launch_straddling(hipStream_t stream, const ConvTileArgs &g, const Epilogue &epilogue)
	{
		if (g.k_bytes == 0) /* as above */
			return false;
		if (try_launch_small_tiles<T, ConvOrder::STRADDLING>(stream, g, epilogue))
			return true;
		if (stays_register_staged(g, sizeof(T)))
			return false;
		launch_conv_tiles_as<T, ConvTile128x64, ConvOrder::STRADDLING>(stream, g, epilogue);
		return true;
	}
} /* namespace mlhip */

#endif /* MINML_AMD_CONV_TILES_HPP_ */
