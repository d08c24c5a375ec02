"""The encoder half of SamPredictor (segment_anything_fast/predictor.py:17-91).

`set_torch_image` keeps its contract - a (B, 3, H, W) image whose long side equals
the encoder input size is normalised, padded and encoded, and the embedding is
kept in `self.features` - so code that drives the image encoder through the
predictor runs unchanged.  Prompt decoding (`predict`, `predict_torch`) belongs
to the mask decoder, which this package does not contain.
"""

from typing import Optional, Tuple

import torch

from . import ops
from .graphs import ReplayedEncoder
from .modeling import Sam


class SamPredictor:
    def __init__(self, sam_model: Sam) -> None:
        self.model = sam_model
        self.reset_image()

    @property
    def device(self) -> torch.device:
        return self.model.device

    def reset_image(self) -> None:
        self.is_image_set = False
        self.features = None
        self.orig_h = self.orig_w = None
        self.input_h = self.input_w = None
        self.original_size = None
        self.input_size = None

    @torch.no_grad()
    def set_torch_image(self, transformed_image: torch.Tensor,
                        original_image_size: Tuple[int, ...]) -> None:
        size = self.model.image_encoder.img_size
        assert (transformed_image.dim() == 4 and transformed_image.shape[1] == 3
                and max(transformed_image.shape[2:]) == size), \
            f"set_torch_image input must be BCHW with long side {size}."
        self.reset_image()
        self.original_size = original_image_size
        self.input_size = tuple(transformed_image.shape[-2:])
        encoder = self.model.image_encoder
        dtype = next(encoder.parameters()).dtype
        self.features = self._encoded(transformed_image, size, dtype)
        self.is_image_set = True

    def _encoded(self, image: torch.Tensor, size: int, dtype: torch.dtype) -> torch.Tensor:
        encoder = self.model.image_encoder
        if isinstance(encoder, ReplayedEncoder):
            with encoder.turn:
                buffer = encoder.input_buffer((image.shape[0], 3, size, size), dtype, image.device)
                if buffer is not None and self._preprocessed(image, size, dtype, buffer) is buffer:
                    return encoder(buffer)
        x = self._preprocessed(image, size, dtype)
        return encoder(self.model.preprocess(image).to(dtype) if x is None else x)

    def _preprocessed(self, image: torch.Tensor, size: int, dtype: torch.dtype, buffer: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
        """The encoder's input in one launch, in `buffer` where given; None where the model's own preprocess has to run (a class
        of its own, a method put in its place, an input the kernel does not read)."""
        model = self.model
        if type(model).preprocess is not Sam.preprocess or "preprocess" in model.__dict__:
            return None
        return ops.preprocess(image, model.pixel_mean, model.pixel_std, size, dtype, buffer)

    def get_image_embedding(self) -> torch.Tensor:
        if not self.is_image_set:
            raise RuntimeError("An image must be set with .set_image(...) to generate an embedding.")
        return self.features

    def predict(self, *args, **kwargs):
        raise NotImplementedError("mask decoding is not part of samfast_amd")

    predict_torch = predict
